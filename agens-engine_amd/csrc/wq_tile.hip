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

// The launch shape with the smallest estimated time (rb = 0: none fits).  Workgroups run in rounds of one per CU; a split
// takes as long as its longest stripe: 9 tiles are 2 per stripe, not 9 / 8.
// Up to two token tiles, and at group 64, a step (one group of inputs) takes about 0.45 + 0.21 rb us, three quarters of
// that at group 64, two workgroups of up to 2 blocks share a CU at about 0.85 of the time, and a split adds its partials'
// traffic (2 us per 4 MB, 2.5 at group 64) and the last workgroups' sums (90000 x 9216 W4 g64, 1 token: split 211, unsplit
// 140; 98304 x 8192 W4 g64, 1 token: split 151, unsplit 130).
// From three token tiles on at group 128 (fitted to 10000 calls of 33 to 128 tokens) a step takes 0.43 + 0.168 rb us, 7 %
// more at W3; 2 blocks from five token tiles on, where the unsplit W4 and W3 kernels spill, up to 0.33 more; two workgroups
// of 2 blocks share a CU where the LDS holds both, at 3 and 5 token tiles.  Every round costs its start and its end: 3 us
// unsplit, 1.6 per block and wave split, where each workgroup stores its partials and waits for them.  (With the estimate
// for up to two token tiles there, splits of several rounds were taken that are slower: 22288 x 6528 W3 at 64 tokens 104 us
// in 3 rounds, 71 unsplit; 12635 x 6912 W3 75 in 2, 50; 11275 x 7296 W2 at 49 68 in 2, 48.)
// So wide linears run unsplit with the most blocks per wave that do not start another round, narrow ones split k at the size
// that fills one, and in between unsplit launches that leave CUs idle are often faster than split ones of several rounds.
// Measured (us):
//   gate_up 55296 x 5120 W3, 64 tokens: 7 blocks (247 workgroups) 86, 5 (346) 132, 4 (432) 103;
//   down 5120 x 27648 W2, 64 tokens, split: 5 blocks (256 workgroups) 60, 4 (320) 92, 2 (640) 88;
//   o 5120 x 5120 W4, 64 tokens: split 4 blocks (200) 28.8, 2 (400) 32.2, unsplit 2 blocks (80) 35.1;
//   head 152064 x 5120 W4 g64, 1 token: 2 blocks (594) 126, 1 (1188) 180.
TileShape pick_shape(const TileArgs& a, int group, int bits) {
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
      const double steps = (sk ? (ntile + a.P - 1) / a.P : ntile) * (1024.0 / group) * (group == 64 ? 0.75 : 1.0);
      const double part = sk ? 1024 / 4e6 * a.P * blocks * a.ntt : 0.0;  // 4 MB of partials
      double us;
      if (group == 64 || a.ntt <= 2) {
        us = rounds * (t.rb <= 2 && rounds > 1 ? 0.85 : 1.0) * steps * (0.45 + 0.21 * t.rb) +
             (sk ? 4.0 + (group == 64 ? 2.5 : 2.0) * part : 0.0);
      } else {
        const bool pair = t.rb <= 2 && rounds > 1 && 2 * tile_lds(t, group, a.ntt) <= 160 * 1024;
        const double spill = a.ntt <= 4 || t.rb > 2 ? 0.0 : sk ? 0.12 : bits == 2 ? 0.06 : bits == 3 ? 0.27 : 0.33;
        const double step = (0.43 + 0.168 * t.rb) * (bits == 3 ? 1.07 : 1.0) + spill;
        us = rounds * (steps * step * (pair ? 0.85 : 1.0) + (sk ? 1.6 * t.rb : 3.0)) +
             (sk ? 8.0 + 1.5 * part : 5.0);
      }
      if (us < best_us) best_us = us, best = t;
    }
  return best;
}

// 33 to 40 tokens at group 128 and k > 10240, where the other side is the integer kernels (wq_i8mt.hip) in chunks of 16
// tokens, the third a short one: they are the faster ones where this kernel is split over more than one round, or unsplit
// leaves three eighths of the CUs idle (a quarter from 14 tiles of inputs on), with one or two tiles per stripe, at W2 with
// more too, but for up to about 10000 rows, where the two are equal.  Measured (us, tiled / integer, 33 tokens): split 10600
// x 16384 W2 88 / 75, 11689 x 13312 W4 88 / 79, 17192 x 15872 W3 131 / 116, 8192 x 10496 W4 61 / 58; unsplit 17835 x 12928 W4
// 127 / 108, 22614 x 15872 W2 150 / 126, but 22000 x 10496 W4 108 / 121, 16000 x 10496 W2 (250 workgroups) 73 / 87; more
// tiles per stripe 10597 x 21248 W2 112 / 96, 12288 x 19712 W3 123 / 133, 18000 x 27648 W4 212 / 237; fewer inputs 22000 x
// 8448 W4 89 / 122.  41 to 48 tokens take 0.92 to 1.04 of the integer kernels' time.
bool integer_kernels_faster(const TileArgs& a, const TileShape& t, int bits, int k, int group) {
  if (group != 128 || k <= 10240 || a.m <= 32 || a.m > 40) return false;
  const int ranges = row_ranges(a.segs, t.rg * t.rb), cus = num_cus(), ntile = kpad(k) / 1024;
  if (t.sk ? ranges * a.P <= cus : 8 * ranges >= (ntile >= 14 ? 6 : 5) * cus) return false;
  long long rows = 0;
  for (int i = 0; i < a.segs.nseg; ++i) rows += a.segs.n[i];
  return rows > 10240 && (bits == 2 || ntile <= 2 * a.P);
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
  const TileShape t = pick_shape(a, group, bits);
  if (!t.rb || integer_kernels_faster(a, t, bits, k, group)) return AK_INVALID;
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
