// The batched default-numerics GEMV (speculative verify, batched decode; groups of 128 and 64) on gfx950 as a tiled
// integer product: the activations are converted once per call, every weight is read and unpacked once per call, and
// 16-token tiles share it.
//
// Numerics: the default numerics (wq_i8.hip), bit for bit, like every other kernel of that route: exact integer group sums
// on v_mfma_i32_16x16x64_i8, one rounding to fp32 per group, the same fp32 order (four group-slot sums per stripe, then
// ((a0 + a1) + a2) + a3, then the stripes).
//
// What bounded the older routes was the conversions: at more than 16 tokens every workgroup of wq_mm.hip converts the
// activations for itself, and again for every 32 tokens, for which it also reads and unpacks the weights again; the
// any-m kernel (all that group 64 had) converts and unpacks per 2 tokens.  Here
//   - a first launch (4 to 5 us) writes the activations' int8 limbs, in MFMA operand order, with their bias and scale:
//     the GEMM loads them straight into LDS, 1 KB per instruction;
//   - a workgroup holds all tokens of its rows (8 waves = token tiles x row groups), so a weight is unpacked once, into
//     LDS, double-buffered, and read as an operand by the waves of every token tile;
//   - requests run ahead of their use (records 1 to 2 steps, weights 2 to 4, scales a 1024-input tile) under counted
//     waits, and one block's products are issued while the block before is rounded and added;
//   - groups are walked in memory order, so a cache line of weights is used up within 2 to 4 steps (walking slot by
//     slot, with a quarter of the accumulators, left each line to be fetched up to four times from beyond the L2:
//     152064 x 5120 W4 g64 214 us, now 126).
// Measured (us, older route -> this): 55296 x 5120 W3 at 64 tokens 163 -> 86 (VALU half busy: the rounding of 4 outputs
// per lane and product; MFMA 30 %; LDS a third), at 128 324 -> 150, at 32 82 -> 60; 5120 x 27648 W2 at 37 78 -> 60;
// group 64, 5120 x 6144 W4 at 2 tokens 29.8 -> 18.4, at 16 188 -> 18.9.
#pragma once
#include "agens_kernels.h"
#include "wq_common.h"
#include "wq_i8_common.h"

#include <type_traits>

namespace agq {

int num_cus();

struct TileArgs {
  Segs segs;
  const uint8_t* img;  // activation image: [group][token tile] records (tile_rec_bytes)
  size_t img_bytes;
  float* part;      // SK: stripe partials [P][16-row blocks][16 ntt tokens][16 rows] per segment
  int* cnt;         // SK: one counter per row range
  int m, ntt;       // tokens, 16-token tiles
  int nquad, P;     // quads (4 groups) of inputs, stripes
  unsigned pmul;    // x / P as a multiplication (upto8_mul; 0 for P = 1)
  int wg_end[4];    // workgroups (SK: x P) of segments 0..i
};

// one token tile's record of one group: limbs [3][MFMA halves][64 lanes][16 B], then the bias -OFF * sum(d_j) [3][16
// tokens] int32 and the activation scale [16] fp32
__host__ __device__ constexpr int tile_img_bytes(int group) { return group * 48; }
__host__ __device__ constexpr int tile_rec_bytes(int group) { return tile_img_bytes(group) + 256; }

// a launch's shape: rg x (8 / rg) waves per workgroup (row groups x token tiles), rb 16-row blocks per wave, split-K
struct TileShape {
  int rg, rb;
  bool sk;
};
__host__ __device__ constexpr int tile_stages(int rg) { return rg == 1 ? 2 : 3; }  // LDS stages of activation records
// bytes of one 1024-input tile's scales of `blocks` 16-row blocks, in whole 1 KB loads
__host__ __device__ constexpr int tile_scale_stage(int blocks, int group) {
  return (blocks * 16 * (2048 / group) + 1023) & ~1023;
}
// LDS of a launch: two stages of unpacked weights and of scales, the activation records
inline size_t tile_lds(const TileShape& t, int group, int ntt) {
  return 2 * (size_t)t.rg * t.rb * group * 16 + 2 * (size_t)tile_scale_stage(t.rg * t.rb, group) +
         (size_t)tile_stages(t.rg) * ((ntt * tile_rec_bytes(group) + 1023) & ~1023);
}

namespace {

constexpr int kRsrcWord3 = 0x00020000;  // raw buffer resource, dword 3 (CDNA)
constexpr int kVmcnt0 = 0x0F70;         // s_waitcnt immediate: vector memory counter 0, the others unconstrained

// the workgroup meets with at most N of each wave's global loads outstanding and its LDS accesses done (a fence would
// wait for every load into LDS in flight)
template <int N>
__device__ __forceinline__ void wait_barrier() {
  static_assert(N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// input (of a 32-input lane chunk) whose limb byte lands in half hf, dword v, byte b of the MFMA operand (make_b)
template <int BITS>
__host__ __device__ constexpr int tile_pos(int hf, int v, int b) {
  return BITS == 4 ? 8 * v + 2 * b + hf : BITS == 2 ? 16 * hf + 4 * b + v : 8 * b + 4 * hf + v;
}

// f(integral_constant<int, I>) for I = B .. E - 1, unrolled at compile time
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>());
    static_for<B + 1, E>(f);
  }
}

// The activation image: one wave per (128 inputs, token tile), lane (c, h) = token c, 32-input chunk h.  act: x is the
// merged gate_up [m][2k] and the activations are SiLU(gate) * up (wq_silu.h).  Padding (tokens past m, inputs past k)
// converts as zeros.
template <int BITS, int G>
__global__ void __launch_bounds__(256) tile_image_kernel(const uint16_t* __restrict__ x, int m, int k, int ntt, int act,
                                                         int n128, uint8_t* __restrict__ img) {
  constexpr int REC = tile_rec_bytes(G), IMG = tile_img_bytes(G), OFF = code_offset<BITS>();
  const int id = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, c = lane & 15, h = lane >> 4;
  if (id >= n128 * ntt) return;
  const int g128 = id / ntt, tt = id - g128 * ntt, t = tt * 16 + c, i0 = g128 * 128 + 32 * h;
  const bool in = t < m && i0 < k;
  const uint4* xp = reinterpret_cast<const uint4*>(x + (in ? (size_t)t * (act ? 2 * (size_t)k : (size_t)k) + i0 : 0));
  uint32_t X[16];
  uint32_t mx = 0;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    uint4 d = xp[v];
    if (act) d = silu_mul8(d, *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(xp + v) + (in ? k : 0)));
    X[4 * v] = in ? d.x : 0u, X[4 * v + 1] = in ? d.y : 0u, X[4 * v + 2] = in ? d.z : 0u, X[4 * v + 3] = in ? d.w : 0u;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) mx = max(mx, max(X[i] & 0x7FFFu, (X[i] >> 16) & 0x7FFFu));
  int mxi = (int)mx;
  mxi = max(mxi, __shfl_xor(mxi, 16));
  if (G == 128) mxi = max(mxi, __shfl_xor(mxi, 32));
  const XiScale xs = xi_scale(mxi >> 7);
  uint32_t xi[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) xi[i] = (uint32_t)x_int((X[i >> 1] >> (16 * (i & 1))) & 0xFFFFu, xs);
  const int g = G == 128 ? g128 : 2 * g128 + (h >> 1);
  uint8_t* rec = img + ((size_t)g * ntt + tt) * REC;
  int sum[3] = {0, 0, 0};
#pragma unroll
  for (int limb = 0; limb < 3; ++limb) {
    const uint32_t add = limb == 0 ? 0u : limb == 1 ? 0x80u : 0x8080u;
    const uint32_t sel = (uint32_t)limb | ((uint32_t)(4 + limb) << 8) | 0x0C0C0000u;  // [a.byte l, b.byte l, 0, 0]
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      uint32_t d[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const uint32_t lo = __builtin_amdgcn_perm(xi[tile_pos<BITS>(hf, v, 1)] + add, xi[tile_pos<BITS>(hf, v, 0)] + add, sel);
        const uint32_t up = __builtin_amdgcn_perm(xi[tile_pos<BITS>(hf, v, 3)] + add, xi[tile_pos<BITS>(hf, v, 2)] + add, sel);
        d[v] = lo | (up << 16);
        sum[limb] = __builtin_amdgcn_sdot4((int)d[v], 0x01010101, sum[limb], false);
      }
      const int slot = G == 128 ? hf * 64 + lane : ((h & 1) + 2 * hf) * 16 + c;
      *reinterpret_cast<uint4*>(rec + limb * (IMG / 3) + slot * 16) = make_uint4(d[0], d[1], d[2], d[3]);
    }
  }
#pragma unroll
  for (int limb = 0; limb < 3; ++limb) {
    sum[limb] += __shfl_xor(sum[limb], 16);
    if (G == 128) sum[limb] += __shfl_xor(sum[limb], 32);
  }
  if (G == 128 ? h == 0 : (h & 1) == 0) {
    int* meta = reinterpret_cast<int*>(rec + IMG);
#pragma unroll
    for (int limb = 0; limb < 3; ++limb) meta[limb * 16 + c] = -OFF * sum[limb];
    meta[48 + c] = act_scale_bits(mxi);
  }
}

// the group's limb sums -> fp32_rn of the group sum (group_sum_f32; W2 / W3: the sum itself fits 32 bits, |x_int| < 2^22,
// |q| <= 4, 128 inputs, and one conversion rounds it)
template <int BITS>
__device__ __forceinline__ float tile_group_sum(int d0, int d1, int d2) {
  if constexpr (BITS == 4)
    return fmaf((float)(d2 * 256 + d1), 256.0f, (float)d0);
  else {
    int t = d2 * 256 + d1;
    asm("" : "+v"(t));  // two shift-adds, not two shifts and an add of three
    return (float)(t * 256 + d0);
  }
}

// LDS slot (16 bytes) of lane group h's operand of row r within a block: the rows of group h are permuted by an xor with
// -4 h, so that neither the operand reads (one row per lane) nor the unpacking's writes (all groups of a row side by
// side) put two lanes of a 16-lane pass (lanes 0-3, 12-15, 20-23, 24-27 and so on) on the same banks
__device__ __forceinline__ int tile_slot(int h, int r) { return h * 16 + (r ^ ((-4 * h) & 15)); }

// RG x TW = 8 waves: wave = token tile (wave % TW), row group (wave / TW) of RB 16-row blocks.  NA: LDS stages of the
// activation records; R: register sets of raw weights.  SK: workgroup = (row range, stripe).  RB <= 2 is held to 128
// registers so that two workgroups fit a CU (up to RB = 2 at 2, 3 and 5 token tiles of group 128; at 4 and 6 to 8 the LDS
// holds one, and the bound only makes the unsplit kernels spill: W4 3 registers at RG = 2 and 15 at RG = 1, W3 1 and 4).
template <int BITS, int G, int RG, int RB, bool SK>
__global__ void __launch_bounds__(512, RB <= 2 ? 4 : 2) tile_kernel(const TileArgs a) {
  constexpr int NW = 8, NT = 512, TW = NW / RG, NA = tile_stages(RG), R = RB >= 5 ? 2 : 4;
  constexpr int REC = 128 * BITS, AREC = tile_rec_bytes(G), AIMG = tile_img_bytes(G);
  constexpr int CH = G / 32, NCH = RG * RB * 16 * CH, CPT = (NCH + NT - 1) / NT;  // lane chunks per step, per thread
  constexpr int BBLK = G * 16, BSTAGE = RG * RB * BBLK, SROW = 2048 / G, SSTAGE = tile_scale_stage(RG * RB, G);
  constexpr int DPW = (TW * AREC + NW * 1024 - 1) / (NW * 1024);                 // 1 KB record blocks per wave and step
  constexpr int WL = CPT * (BITS == 3 ? 2 : 1);                  // weight loads per step
  constexpr int QPT = 256 / G;                                   // quads per 1024-input tile
  constexpr int CB = BITS == 4 ? 16 : 8;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  uint8_t* const ldsb = lds;                       // [2] weight stages (int8 codes in operand order)
  uint8_t* const ldss = lds + 2 * BSTAGE;          // scales (bf16) [tile parity]
  uint8_t* const ldsa = ldss + 2 * SSTAGE;      // [NA] activation records
  const int ntt = a.ntt, astage = (ntt * AREC + 1023) & ~1023, ablk = astage >> 10;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, h = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), tt = wave % TW, rgi = wave / TW;
  const bool busy = tt < ntt;
  const Segs& sgs = a.segs;
  const int P = a.P, nquad = a.nquad;

  int sg = 0;
#pragma unroll
  for (int i = 1; i < kMaxSegs; ++i) sg += (i < sgs.nseg && (int)blockIdx.x >= a.wg_end[i - 1]) ? 1 : 0;
  auto pick = [&](auto v0, auto v1, auto v2, auto v3) { return sg == 0 ? v0 : sg == 1 ? v1 : sg == 2 ? v2 : v3; };
#define AK_SEG(arr) pick((arr)[0], (arr)[1], (arr)[2], (arr)[3])
  const int wg0 = sg ? (sg == 1 ? a.wg_end[0] : sg == 2 ? a.wg_end[1] : a.wg_end[2]) : 0;
  const int li = (int)blockIdx.x - wg0, rr_ = SK ? li / P : li, psk = SK ? li - rr_ * P : 0;
  const int n = AK_SEG(sgs.n), n_b16 = (n + 15) >> 4, ldy = AK_SEG(sgs.ldy);
  uint16_t* const yseg = AK_SEG(sgs.y);
  const int row0 = rr_ * RG * RB * 16;  // first row of the workgroup
  const int pa = SK ? psk : 0, pb = SK ? psk + 1 : P;

  // ---- loads of a step: the group's lane chunks of the workgroup's rows, and the scales
  const int ntile = nquad / QPT;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(AK_SEG(sgs.wt)), (short)0,
                                                                      ntile * n * REC, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(AK_SEG(sgs.st)), (short)0,
                                                                      ntile * n * (2048 / G), kRsrcWord3);
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.img), (short)0, (int)a.img_bytes, kRsrcWord3);
  int vw[CPT], dst[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int idx = tid + NT * j, row = idx / CH, ch = idx % CH;
    const int o = row0 + row < n ? row0 + row : n - 1;
    vw[j] = o * REC + ch * CB;
    const int rr = row & 15, hp = G == 128 ? ch : ch & 1;
    dst[j] = idx < NCH ? (row >> 4) * BBLK + tile_slot(hp, rr) * 16 : -1;
  }
  const int vhd = (lane % CH) * (4 - CB) + 256;  // third-bit word of the chunk, relative to vw
  auto begin = [&](int p) __attribute__((always_inline)) {  // first quad of stripe p
    const int x = p * ntile;
    return QPT * ((int)(((unsigned long long)(unsigned)x * a.pmul) >> 32) + (P == 1 ? x : 0));
  };
  struct Set {
    Raw<BITS> r[CPT];
  };
  Set raw[R];
  auto fetch = [&](int g, Set& d) __attribute__((always_inline)) {
    const int t = g / (4 * QPT), gt = g % (4 * QPT), tb = t * n * REC;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      if constexpr (BITS == 4) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rw, vw[j], tb + gt * CH * CB, 0);
        d.r[j].w = make_uint4(v[0], v[1], v[2], v[3]);
      } else {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, vw[j], tb + gt * CH * CB, 0);
        d.r[j].lo = make_uint2(v[0], v[1]);
        if constexpr (BITS == 3) d.r[j].hi = __builtin_amdgcn_raw_buffer_load_b32(rw, vw[j] + vhd, tb + gt * CH * 4, 0);
      }
    }
  };
  auto dma = [&](int g, int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < DPW; ++j) {
      const int b = wave + NW * j < ablk ? wave + NW * j : ablk - 1;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ra, (__attribute__((address_space(3))) void*)(ldsa + stage * astage + b * 1024), 16, lane * 16,
          g * ntt * AREC + b * 1024, 0, 0);
    }
  };
  // the scales of tile t into scale stage ss.  Blocks that start past the segment's last row are left out: the scalar
  // offset stays within the buffer, whose end then bounds the lanes
  const int sblk = min(SSTAGE / 1024 - 1, (n - 1 - row0) * SROW / 1024);
  auto dma_scales = [&](int t, int ss) __attribute__((always_inline)) {
    if (t >= ntile) t = ntile - 1;  // (past the end: read again, not used)
#pragma unroll
    for (int j = 0; j < (SSTAGE / 1024 + NW - 1) / NW; ++j) {
      int b = wave + NW * j;
      if (b > sblk) b = sblk;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (__attribute__((address_space(3))) void*)(ldss + ss * SSTAGE + b * 1024), 16, lane * 16,
          (t * n + row0) * SROW + b * 1024, 0, 0);
    }
  };
  auto put = [&](const Set& d, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      i32x4 b0, b1;
      make_b<BITS>(d.r[j], b0, b1);
      if (NCH % NT == 0 || dst[j] >= 0) {
        uint8_t* p = ldsb + st * BSTAGE + dst[j];
        *reinterpret_cast<i32x4*>(p) = b0;
        if constexpr (G == 128) {
          *reinterpret_cast<i32x4*>(p + 1024) = b1;
        } else {  // half 1: lane groups 2, 3
          const int row = (tid + NT * j) / CH, hp = ((tid + NT * j) & 1) + 2;
          *reinterpret_cast<i32x4*>(ldsb + st * BSTAGE + (row >> 4) * BBLK + tile_slot(hp, row & 15) * 16) = b1;
        }
      }
    }
  };

  // sums of the stripe's groups by slot (group % 4) and, unsplit, the sum of the finished stripes
  float acc[4][RB][4], yv[SK ? 1 : RB][4];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int s = 0; s < 4; ++s) acc[s][b][i] = 0.f;
      if constexpr (!SK) yv[b][i] = 0.f;
    }
  const int rdb = rgi * RB * BBLK + tile_slot(h, c) * 16, rds = (rgi * RB * 16 + c) * SROW;

  // the step's products: all row blocks of this wave against its token tile
  auto compute = [&](auto UU, int as, int so) __attribute__((always_inline)) {
    constexpr int slot = decltype(UU)::value, st = slot & 1;
    const uint8_t* rec = ldsa + as * astage + tt * AREC;
    i32x4 A[3][G / 64], C[3];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
#pragma unroll
      for (int hf = 0; hf < G / 64; ++hf)
        A[l][hf] = *reinterpret_cast<const i32x4*>(rec + l * (AIMG / 3) + hf * 1024 + lane * 16);
      C[l] = *reinterpret_cast<const i32x4*>(rec + AIMG + l * 64 + h * 16);
    }
    // (read as integers: the compiler orders an LDS read of another type behind the record loads in flight)
    const i32x4 xe = *reinterpret_cast<const i32x4*>(rec + AIMG + 192 + h * 16);
    const float xev[4] = {__int_as_float(xe[0]), __int_as_float(xe[1]), __int_as_float(xe[2]), __int_as_float(xe[3])};
    // block b's operands are read and its products issued while block b - 1's are rounded and added
    i32x4 B[2][G / 64], D[2][3];
    float sc[2];
    auto read = [&](auto BB) __attribute__((always_inline)) {
      constexpr int b = decltype(BB)::value;
#pragma unroll
      for (int hf = 0; hf < G / 64; ++hf)
        B[b & 1][hf] = *reinterpret_cast<const i32x4*>(ldsb + st * BSTAGE + rdb + b * BBLK + hf * 1024);
    };
    read(std::integral_constant<int, 0>());
    static_for<0, RB + 1>([&](auto BB) __attribute__((always_inline)) {
      constexpr int b = decltype(BB)::value, e = b - 1;  // the block whose products are issued, and rounded
      if constexpr (b < RB) {
        sc[b & 1] = bf2f(*reinterpret_cast<const uint16_t*>(ldss + so + rds + b * 16 * SROW));
        if constexpr (b + 1 < RB) read(std::integral_constant<int, b + 1>());
#pragma unroll
        for (int l = 0; l < 3; ++l) D[b & 1][l] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[l][0], B[b & 1][0], C[l], 0, 0, 0);
        if constexpr (G == 128)
#pragma unroll
          for (int l = 0; l < 3; ++l)
            D[b & 1][l] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[l][1], B[b & 1][G / 64 - 1], D[b & 1][l], 0, 0, 0);
      }
      if constexpr (e >= 0) {
        constexpr int o = e & 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float gs = tile_group_sum<BITS>(D[o][0][i], D[o][1][i], D[o][2][i]), sx = sc[o] * xev[i];
          acc[slot][e][i] = fmaf(gs, sx, acc[slot][e][i]);
        }
      }
      if constexpr (b > 0 && b < RB) {
        static_for<0, 3 * (G / 64)>([&](auto) __attribute__((always_inline)) {
          __builtin_amdgcn_sched_group_barrier(0x0100, 1, 0);                       // DS read
          __builtin_amdgcn_sched_group_barrier(0x0008, 1, 0);                       // MFMA
          __builtin_amdgcn_sched_group_barrier(0x0002, G == 128 ? 4 : 8, 0);        // VALU
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto stripe_sum = [&](int b, int i) __attribute__((always_inline)) {
    return ((acc[0][b][i] + acc[1][b][i]) + acc[2][b][i]) + acc[3][b][i];
  };

  // ---- pipeline: step i computes stage i; meanwhile the weights of step i + 1 are unpacked into the other stage, the
  // records of step i + NA - 1 and the raw weights of step i + R are requested.  The barrier at the end of a step waits
  // for the records of the next (by count: what was requested after them stays in flight)
  const int q0 = begin(pa), q1 = begin(pb), g_end = 4 * q1 - 1;
  auto head = [&](int g, Set& d) __attribute__((always_inline)) { fetch(min(g, g_end), d); };
  int sd = NA - 1, sa = 0;
  static_for<0, R>([&](auto U) __attribute__((always_inline)) { head(4 * q0 + decltype(U)::value, raw[decltype(U)::value]); });
#pragma unroll
  for (int i = 0; i < NA - 1; ++i) dma(4 * q0 + i, i);
  dma_scales(q0 / QPT, (q0 / QPT) & 1);
  put(raw[0], 0);
  wait_barrier<0>();
  auto step = [&](auto U, int g, int so) __attribute__((always_inline)) {
    constexpr int u = decltype(U)::value, st = u & 1;
    __builtin_amdgcn_sched_barrier(0);
    dma(min(g + NA - 1, g_end), sd);
    __builtin_amdgcn_sched_barrier(0);
    head(g + R, raw[u % R]);
    sd = sd + 1 == NA ? 0 : sd + 1;
    __builtin_amdgcn_sched_barrier(0);
    if (busy) compute(U, sa, so + 2 * u);
    put(raw[(u + 1) % R], st ^ 1);
    sa = sa + 1 == NA ? 0 : sa + 1;
    __builtin_amdgcn_sched_barrier(0);
    wait_barrier<(NA - 2) * (DPW + WL) + WL>();
  };
  int p = pa, qe = begin(pa + 1);
  for (int q = q0; q < q1; ++q) {
    // the next tile's scales, a tile ahead; the steps' counted waits cover them long before their first use
    const int t = q / QPT, so = (t & 1) * SSTAGE + (q % QPT) * 8;
    if (q % QPT == 0) dma_scales(t + 1, (t + 1) & 1);
    step(std::integral_constant<int, 0>(), 4 * q, so);
    step(std::integral_constant<int, 1>(), 4 * q + 1, so);
    step(std::integral_constant<int, 2>(), 4 * q + 2, so);
    step(std::integral_constant<int, 3>(), 4 * q + 3, so);
    if constexpr (!SK)
      if (q + 1 == qe) {
        ++p;
        qe = begin(p + 1);
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            yv[b][i] += stripe_sum(b, i);
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[s][b][i] = 0.f;
          }
      }
  }
  __builtin_amdgcn_s_waitcnt(kVmcnt0);  // no load into LDS outlives the loop

  if constexpr (!SK) {
    if (busy) {
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const int row = row0 + (rgi * RB + b) * 16 + c;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = tt * 16 + 4 * h + i;
          if (row < n && t < a.m) yseg[(size_t)t * ldy + row] = f2bf(yv[b][i]);
        }
      }
    }
  } else {
    // the stripe's partials to scratch, device-coherent; every store is acknowledged before the range's counter moves;
    // the range's last workgroup adds the P partials of each output in stripe order
    const int MP = 16 * ntt, blk0 = row0 >> 4;
    float* spart = a.part;
    int* scnt = a.cnt + wg0 / P + rr_;
#pragma unroll
    for (int i = 0; i < kMaxSegs - 1; ++i)
      if (i < sg) spart += (size_t)P * MP * ((sgs.n[i] + 15) >> 4) * 16;
    if (busy) {
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const int blk = blk0 + rgi * RB + b;
        if (blk < n_b16)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            __hip_atomic_store(spart + (((size_t)psk * n_b16 + blk) * MP + tt * 16 + 4 * h + i) * 16 + c, stripe_sum(b, i),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __builtin_amdgcn_s_waitcnt(kVmcnt0);
    __syncthreads();
    int* const last = reinterpret_cast<int*>(lds);
    if (tid == 0) {
      const int old = __hip_atomic_fetch_add(scnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = old == P - 1;
      if (old == P - 1) __hip_atomic_store(scnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next launch
    }
    __syncthreads();
    if (!*last) return;
    const int nb = n_b16 - blk0 < RG * RB ? n_b16 - blk0 : RG * RB, ne = nb * MP * 16;
    for (int i0 = tid; i0 < ne; i0 += 2 * NT) {
      const size_t off[2] = {(size_t)blk0 * MP * 16 + i0, (size_t)blk0 * MP * 16 + (i0 + NT < ne ? i0 + NT : i0)};
      float y[2];
      sum_stripe_partials_n<2>(spart, off, (size_t)MP * n_b16 * 16, P, y);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int i = i0 + u * NT, bl = i / (MP * 16), o = i - bl * MP * 16, t = o >> 4;
        const int row = (blk0 + bl) * 16 + (o & 15);
        if (i < ne && t < a.m && row < n) yseg[(size_t)t * ldy + row] = f2bf(y[u]);
      }
    }
  }
#undef AK_SEG
}

template <int BITS, int G>
int tile_launch(const TileArgs& a, const TileShape& t, const void* x, int k, int act, uint8_t* img, hipStream_t s) {
  const int n128 = kpad(k) / 128, waves = n128 * a.ntt;
  hipLaunchKernelGGL((tile_image_kernel<BITS, G>), dim3((waves + 3) / 4), dim3(256), 0, s,
                     static_cast<const uint16_t*>(x), a.m, k, a.ntt, act, n128, img);
  if (const int e = (int)hipGetLastError()) return e;
  const dim3 grid(a.wg_end[a.segs.nseg - 1]);
  const size_t smem = tile_lds(t, G, a.ntt);
#define AK_TILE(RG, RB)                                                                                         \
  case RG * 100 + RB * 10:                                                                                      \
    hipLaunchKernelGGL((tile_kernel<BITS, G, RG, RB, false>), grid, dim3(512), smem, s, a);                     \
    return (int)hipGetLastError();                                                                              \
  case RG * 100 + RB * 10 + 1:                                                                                  \
    hipLaunchKernelGGL((tile_kernel<BITS, G, RG, RB, true>), grid, dim3(512), smem, s, a);                      \
    return (int)hipGetLastError();
  if constexpr (G == 64) {  // (up to 16 tokens at group 128: other kernels)
    switch (t.rg * 100 + t.rb * 10 + (t.sk ? 1 : 0)) { AK_TILE(8, 1) AK_TILE(8, 2) }
  }
  switch (t.rg * 100 + t.rb * 10 + (t.sk ? 1 : 0)) {
    AK_TILE(4, 1) AK_TILE(4, 2) AK_TILE(2, 2) AK_TILE(2, 4) AK_TILE(2, 5) AK_TILE(2, 7) AK_TILE(1, 2) AK_TILE(1, 4)
    AK_TILE(1, 5) AK_TILE(1, 7)
    default: return AK_INVALID;
  }
#undef AK_TILE
}

}  // namespace
}  // namespace agq
