// Host side of the tiled batched GEMV (wq_tile.h): the choice of the launch shape.
#include "wq_tile.h"

namespace agq {

int tile_launch_w2(const TileArgs& a, const TileShape& t, const void* x, int k, int group, int act, uint8_t* img, hipStream_t s);
int tile_launch_w3(const TileArgs& a, const TileShape& t, const void* x, int k, int group, int act, uint8_t* img, hipStream_t s);
int tile_launch_w4(const TileArgs& a, const TileShape& t, const void* x, int k, int group, int act, uint8_t* img, hipStream_t s);

namespace {

int row_ranges(const Segs& g, int blocks) {  // workgroups that cover the segments with `blocks` 16-row blocks each
  int e = 0;
  for (int i = 0; i < g.nseg; ++i) e += ((g.n[i] + 15) / 16 + blocks - 1) / blocks;
  return e;
}

// The launch shape with the smallest estimated time (rb = 0: none fits).  Workgroups run in rounds of one per CU; a step
// (one group of inputs) takes about 0.45 + 0.21 rb us at group 128 and three quarters of that at group 64 (measured us
// per step, g128: 0.65 at 1 block per wave, 0.85 at 2, 1.25 at 4, 1.5 at 5, 1.95 at 7; g64: 0.52 at 1, 0.7 at 2, 1.4 at
// 7), two workgroups of up to 2 blocks per wave share a CU at about 0.85 of the time (applied to every such shape, also
// where the LDS holds only one: group 128 and 2 blocks per wave at 4 and 6 to 8 token tiles).  A split takes as long as its
// longest stripe, and adds its partials' traffic (2 us per 4 MB, 2.5 at group 64) and the last workgroups' sums: 9 tiles
// are 2 per stripe, not 9 / 8 (20000 x 8320 W2, 33 tokens: split 132, unsplit 87; 90000 x 9216 W4 g64, 1 token: 211 and
// 140), and many rows pay more for the partials than for another round (98304 x 8192 W4 g64, 1 token: split 151, unsplit
// 130).  So wide linears run unsplit with the most blocks per wave that do not start another round, narrow ones split k
// at the size that fills one (measured, us):
//   gate_up 55296 x 5120 W3, 64 tokens: 7 blocks (247 workgroups) 86, 5 (346) 132, 4 (432) 103;
//   down 5120 x 27648 W2, 64 tokens, split: 5 blocks (256 workgroups) 60, 4 (320) 92, 2 (640) 88;
//   o 5120 x 5120 W4, 64 tokens: split 4 blocks (200) 28.8, 2 (400) 32.2, unsplit 2 blocks (80) 35.1;
//   head 152064 x 5120 W4 g64, 1 token: 2 blocks (594) 126, 1 (1188) 180.
TileShape pick_shape(const TileArgs& a, int group) {
  static const int kRB[4][4] = {{1, 2, 0, 0}, {1, 2, 0, 0}, {2, 4, 5, 7}, {2, 4, 5, 7}};  // by token tiles per workgroup
  const int w = a.ntt == 1 ? 0 : a.ntt == 2 ? 1 : a.ntt <= 4 ? 2 : 3, rg = 8 >> w;
  const int ntile = a.nquad / (256 / group), cus = num_cus();
  long long blocks = 0;
  for (int i = 0; i < a.segs.nseg; ++i) blocks += (a.segs.n[i] + 15) / 16;
  TileShape best = {rg, 0, false};
  double best_us = 1e30;
  for (int sk = 0; sk < (a.P > 1 ? 2 : 1); ++sk)
    for (int r = 0; r < 4 && kRB[w][r]; ++r) {
      const TileShape t = {rg, kRB[w][r], sk != 0};
      const int ranges = row_ranges(a.segs, rg * t.rb);
      if (tile_lds(t, group, a.ntt) > 160 * 1024 || (sk && ranges > 1024)) continue;
      const long long rounds = ((long long)ranges * (sk ? a.P : 1) + cus - 1) / cus;
      const double steps = (sk ? (ntile + a.P - 1) / a.P : ntile) * (1024.0 / group);
      const double us = rounds * (t.rb <= 2 && rounds > 1 ? 0.85 : 1.0) * steps * (0.45 + 0.21 * t.rb) * (group == 64 ? 0.75 : 1.0) +
                        (sk ? 4.0 + (group == 64 ? 2.5 : 2.0) * 1024 / 4e6 * a.P * blocks * a.ntt : 0.0);
      if (us < best_us) best_us = us, best = t;
    }
  return best;
}

// 33 to 48 tokens at group 128 and k > 8192, where the other side is the integer kernels (wq_i8mt.hip) in chunks of 16
// tokens.  A split launch of more than one round pays 5 to 8 us per round for its start and its partials, which counts
// against stripes of one or two tiles of inputs.  Up to 40 tokens the integer kernels' third chunk is a short one: they are
// faster from two rounds on, at W2 at longer stripes too, but for up to about 10000 rows, where the two are equal.  With a
// full third chunk they are from three rounds on (not with SiLU, which each of their row ranges computes).  Measured (us,
// tiled / integer): 33 tokens, 2 tiles per stripe 11000 x 10496 W4 89 / 73, 18000 x 12544 W3 135 / 113, 14000 x 14592 W2 90
// / 87, 8192 x 10496 W4 61 / 58; 3 and 4 tiles 12288 x 19712 W2 116 / 108, W3 123 / 133, 18000 x 27648 W2 207 / 176, W4 212
// / 237; unsplit 16000 x 10496 W2 73 / 87; 41 tokens 21927 x 13696 W2 155 / 138, 24218 x 14592 W3 172 / 176, 17335 x 11648 W2
// 121 / 112; 42 tokens, two rounds 0.9 of the integer kernels' time, three rounds of 3 tiles 0.7 to 0.9.
bool integer_kernels_faster(const TileArgs& a, const TileShape& t, int bits, int k, int group, int act) {
  if (group != 128 || k <= 8192 || a.m <= 32 || a.m > 48 || !t.sk) return false;
  const int workgroups = row_ranges(a.segs, t.rg * t.rb) * a.P, cus = num_cus();
  const bool short_stripes = kpad(k) / 1024 <= 2 * a.P;
  if (a.m > 40) return workgroups > 2 * cus && short_stripes && !act;
  long long rows = 0;
  for (int i = 0; i < a.segs.nseg; ++i) rows += a.segs.n[i];
  return workgroups > cus && rows > 10240 && (bits == 2 || short_stripes);
}

}  // namespace

// 1..128 tokens at group 64, 17..128 at group 128; act = 1 (group 128): x is the merged gate_up [m][2k] and the activations SiLU(gate) *
// up.  AK_INVALID where the shape does not suit the kernel or there is no scratch for the call (the caller falls back).  Works
// in call_scratch: counters, split-K partials, the activation image; two launches, under scratch_mutex(s).
int tile_gemv(int bits, const void* x, int m, const Segs& g, int k, int group, hipStream_t s, int act) {
  if (group == 128 ? m <= 16 : act) return AK_INVALID;
  TileArgs a;
  a.segs = g;
  a.m = m;
  a.ntt = (m + 15) / 16;
  a.nquad = kpad(k) / group / 4;
  a.P = stripe_count(a.nquad, 256 / group);
  a.pmul = a.P == 1 ? 0u : upto8_mul(a.P);
  for (int i = 0; i < g.nseg; ++i)  // buffer offsets are 32-bit
    if ((long long)(kpad(k) / 1024) * g.n[i] * 128 * bits >= (1ll << 31)) return AK_INVALID;
  a.img_bytes = (size_t)(kpad(k) / group) * a.ntt * tile_rec_bytes(group);
  const TileShape t = pick_shape(a, group);
  if (!t.rb || integer_kernels_faster(a, t, bits, k, group, act)) return AK_INVALID;
  size_t part = 0;
  if (t.sk)
    for (int i = 0; i < g.nseg; ++i) part += (size_t)a.P * a.ntt * ((g.n[i] + 15) / 16) * 1024;
  if (part + a.img_bytes > kMaxCallScratch) return AK_INVALID;  // (128 tokens x 27648 inputs x 5120 rows: 33 MB)
  const CallScratch z = call_scratch(s, part + a.img_bytes);
  if (!z.data) return AK_INVALID;
  a.cnt = z.cnt;
  a.part = reinterpret_cast<float*>(z.data);
  uint8_t* const img = z.data + part;
  a.img = img;
  for (int i = 0, e = 0; i < kMaxSegs; ++i) {
    if (i < g.nseg) e += ((g.n[i] + 15) / 16 + t.rg * t.rb - 1) / (t.rg * t.rb) * (t.sk ? a.P : 1);
    a.wg_end[i] = e;
  }
  return bits == 4   ? tile_launch_w4(a, t, x, k, group, act, img, s)
         : bits == 3 ? tile_launch_w3(a, t, x, k, group, act, img, s)
                     : tile_launch_w2(a, t, x, k, group, act, img, s);
}

}  // namespace agq
