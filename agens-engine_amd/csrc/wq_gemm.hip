// Prefill GEMM straight from the KT weights, gfx950: y[t][o] (row stride ldy) = bf16(sum_i x[t][i] * w[o][i]) with
// w[o][i] = bf16_rn(q * scale) -- the values ak_wq_dequant_kt_rows writes, bit for bit -- and fp32 accumulation.
//
// The reference's prefill route (kernels/m1/m1_model.cu:1876-1897) dequantizes a tile of output rows into a bf16
// scratch (2 bytes per weight written, then read again) and runs a library GEMM (ak_bf16_linear_f32reduce_ld,
// kernels/src/bf16_linear.cu:68-92).  Here the KT records are read once per token tile, expanded to bf16 in registers
// and written to LDS, and v_mfma_f32_32x32x16_bf16 consumes them there: no dequantized copy, no second pass over the
// weights (narrow linears split k across workgroups, with fp32 partials in call_scratch).
//
// Tiling: R = 256 output rows x T tokens (T = 64, 128, 192, 256) per workgroup of 8 waves, or 128 x 128 per workgroup of 4
// (by pick_tiling), wave tiles of 64 rows x T / 2 tokens as 32 x 32 MFMA tiles, k in slabs of 64 inputs.  Thread (row tid / 2, half tid % 2) loads its lane
// chunk of the slab from the row's KT record (W4 16 B, W3 8 + 4 B, W2 8 B) and the group's scale three slabs ahead into
// one of two register sets; the tokens go straight from the buffer into LDS (buffer loads into LDS, two stages, two
// slabs ahead); the weights are dequantized once per T tokens into two LDS stages (32 KB at R = 256).
// What bounds it: per slab a SIMD's two waves need 2048 cycles of MFMA at T = 256, the workgroup's operand reads and
// writes the LDS for as long, and the dequantization about 1400 cycles of each SIMD's VALU; each is hidden behind the
// others only if no wave waits for its own.  So the slab is pipelined in slices of 16 inputs: the operands of a slice (24
// registers with 32 x 32 tiles) are read from LDS while the MFMAs of the slice before run, with a quarter or half of the
// next slab's dequantization mixed in (sched_group_barrier); the slab's barrier stands before its last slice's MFMAs,
// whose operands every wave already holds, so that the next slab's first operands are read behind them and the stage
// just left is free for the DMA of two slabs ahead.  The waits on global loads are counted: the token loads of the next
// slab, not the weights of the one after.
// Measured (us, before = 16 x 16 MFMA tiles with each slice's operands read right before its MFMAs): gate_up 55296 x
// 5120 W3 at 512 tokens 334 -> 283, 300 tokens 326 -> 229 (T = 192), 2048 tokens 1172 -> 1049; o 5120 x 5120 W4 at 256
// tokens 41 -> 31; down 5120 x 27648 W2 at 333 tokens 162 -> 112; 1.0-1.1 PFLOP/s where a round of tiles is full.
// Few tiles (R = 256 only -> with the small tile): 2000 x 1024 W4 at 512 tokens 19.2 -> 13.7, 1000 x 4096 W3 at 512 23.0
// -> 21.3, 3000 x 2048 W2 at 512 28.1 -> 23.8, 14000 x 1024 W3 at 64 19.6 -> 14.2.
// Grid: the items (split, token tile, row tile) in that order cut into 8 contiguous runs, XCD x (workgroup i runs on XCD
// i % 8) taking run x, so that each XCD works on one or two token tiles (T tokens x k inputs) that stay in its L2 while
// the weights stream, and every XCD has as many workgroups as the others.
// Raw buffer loads with a per-lane offset fixed for the kernel and a scalar per-slab offset keep address arithmetic off
// the vector unit; no load sits under a branch (the compiler's wait counts stay exact).  LDS rows / tokens of 64 bf16
// (128 B): the 16-byte chunk q of row r sits at slot q ^ ((r >> 1) & 7), so 16 rows of an MFMA operand read hit 16
// distinct 16-byte bank slots.  Lane l reads 8 inputs 8 (l / 32) .. of its slice for row / token l % 32 (the same
// input-to-slot map for weights and tokens, which is all an MFMA needs).
// The accumulation order is this kernel's own (fp32 MFMA sums over 16 inputs in order, splits in order): results agree with the
// reference's cuBLAS route and with the oracle's dequantized weights times x in fp64 within fp32-accumulation error.
#include <mutex>
#include <type_traits>

#include "agens_kernels.h"
#include "agens_tuning.h"
#include "wq_common.h"

namespace agq {
int num_cus();

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// slabs of 64 inputs (one row / token of a slab: 128 B in LDS), two LDS stages
constexpr int kSlab = 64, kRowBytes = kSlab * 2;
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer resource, dword 3 (CDNA)

// f(integral_constant<int, I>) for I = B .. E - 1, unrolled at compile time
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>());
    static_for<B + 1, E>(f);
  }
}

__device__ __forceinline__ int swz(int r, int q) { return r * kRowBytes + ((q ^ ((r >> 1) & 7)) << 4); }

// the raw bits of one lane chunk (32 inputs) of a KT record and the scale of its group
template <int BITS>
struct ChunkRaw {
  u32x4 w;  // W4: the chunk; W3: lo words in 0, 1 and the third-bit word in 2; W2: lo words in 0, 1
  uint32_t s;
};

// 16 bytes per lane from a buffer straight into LDS: lane l writes dst + 16 l (dst the same for the whole wave)
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}

// the workgroup meets (LDS ordered, loads in flight stay in flight)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 8 codes (one word) -> 8 bf16 bf16_rn((n - OFF) * s): the product is exact in fp32 (an fma of two exact terms), the
// conversion rounds to nearest even
template <int OFF>
__device__ __forceinline__ u32x4 dequant8(uint32_t w, float s) {
  const uint32_t ev = w & 0x0F0F0F0Fu, od = (w >> 4) & 0x0F0F0F0Fu;  // codes of inputs 2b and 2b + 1 in byte b
  const float m = -(float)OFF * s;
  uint32_t o[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const float lo = fmaf((float)((ev >> (8 * b)) & 0xFFu), s, m);
    const float hi = fmaf((float)((od >> (8 * b)) & 0xFFu), s, m);
    const bf16x2 p = {(__bf16)lo, (__bf16)hi};
    o[b] = __builtin_bit_cast(uint32_t, p);
  }
  return u32x4{o[0], o[1], o[2], o[3]};
}

// W2 / W3 without the nibble spread: the 2-bit codes of 16 inputs (one low word of the chunk, input i at bits 2i) as
// four words of byte codes, word p holding inputs 4 j + p in byte j (W3: the third bit, input i at bit i of the high
// half-word, merged at bit 2 of each byte through one 1-to-2 bit spread)
struct HalfCodes {
  uint32_t p0, p1, p2, p3;
};
template <int BITS>
__device__ __forceinline__ HalfCodes half_codes(const ChunkRaw<BITS>& d, int h) {
  const uint32_t L = d.w[h];
  HalfCodes c = {L & 0x03030303u, (L >> 2) & 0x03030303u, (L >> 4) & 0x03030303u, (L >> 6) & 0x03030303u};
  if constexpr (BITS == 3) {
    uint32_t v = (d.w[2] >> (16 * h)) & 0xFFFFu;  // third bits of inputs 16 h .. 16 h + 15; input i -> bit 2 i:
    v = (v | (v << 8)) & 0x00FF00FFu;
    v = (v | (v << 4)) & 0x0F0F0F0Fu;
    v = (v | (v << 2)) & 0x33333333u;
    v = (v | (v << 1)) & 0x55555555u;  // input 4 j + p at bit 8 j + 2 p
    c.p0 |= (v << 2) & 0x04040404u;
    c.p1 |= v & 0x04040404u;
    c.p2 |= (v >> 2) & 0x04040404u;
    c.p3 |= (v >> 4) & 0x04040404u;
  }
  return c;
}
// inputs 8 sub .. 8 sub + 7 of the half as 4 dwords of bf16 pairs bf16_rn((n - OFF) s) (as dequant8)
template <int OFF>
__device__ __forceinline__ u32x4 dequant_half(const HalfCodes& c, float s, int sub) {
  const float m = -(float)OFF * s;
  uint32_t o[4];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    const int sh = 8 * (2 * sub + jj);
    const bf16x2 ab = {(__bf16)fmaf((float)((c.p0 >> sh) & 0xFFu), s, m), (__bf16)fmaf((float)((c.p1 >> sh) & 0xFFu), s, m)};
    const bf16x2 cd = {(__bf16)fmaf((float)((c.p2 >> sh) & 0xFFu), s, m), (__bf16)fmaf((float)((c.p3 >> sh) & 0xFFu), s, m)};
    o[2 * jj] = __builtin_bit_cast(uint32_t, ab);
    o[2 * jj + 1] = __builtin_bit_cast(uint32_t, cd);
  }
  return u32x4{o[0], o[1], o[2], o[3]};
}

// SPLIT: k is split across workgroups; an item's fp32 tile goes to part[item] as its waves hold it (sum_splits_kernel)
template <int BITS, int G, int R, int T, bool SPLIT>
__global__ void __launch_bounds__(2 * R, R == 128 ? 2 : T == 64 ? 4 : 1) wq_gemm_kernel(const uint16_t* __restrict__ x, int m,
                                                              const uint8_t* __restrict__ wt,
                                                              const uint16_t* __restrict__ st,
                                                              uint16_t* __restrict__ y, int n, int ldy, int k,
                                                              int nrow_tiles, int ntok_tiles, int nsplit,
                                                              float* __restrict__ part) {
  constexpr int NW = R / 32, RW = R / 64;             // waves, along the rows
  constexpr int NJ = T / 64, XPW = T / (8 * NW);      // 32-token tiles per wave, 1 KB token blocks per wave and slab
  constexpr int kWStage = R * kRowBytes, kXStage = T * kRowBytes, kXBase = 2 * kWStage;
  constexpr int OFF = BITS == 4 ? 8 : BITS == 3 ? 4 : 2;
  constexpr int REC = 128 * BITS, CB = BITS == 4 ? 16 : 8;
  constexpr int kWLoads = BITS == 3 ? 3 : 2;  // weight and scale loads of a slab
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // workgroup b runs on XCD b % 8 and takes item (b % 8) x per + b / 8: split-major, then token-major tiles, cut into 8
  // contiguous runs
  const int tiles = nrow_tiles * ntok_tiles, items = tiles * nsplit, per = (items + 7) >> 3;
  const int item = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || item >= items) return;
  const int sp = SPLIT ? item / tiles : 0, tile = item - sp * tiles;
  const int tt = tile / nrow_tiles, rt = tile - tt * nrow_tiles;
  const int o0 = rt * R, t0 = tt * T;
  const int sb = SPLIT ? (int)((long long)sp * (k / kSlab) / nsplit) : 0;
  const int nslab = SPLIT ? (int)((long long)(sp + 1) * (k / kSlab) / nsplit) - sb : k / kSlab;

  const int lr = tid >> 1, lj = tid & 1;
  const int orow = o0 + lr < n ? o0 + lr : n - 1;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wt), (short)0, 0x7FFFFFFF,
                                                                      kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(st), (short)0, 0x7FFFFFFF,
                                                                      kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), (short)0, m * k * 2,
                                                                      kRsrcWord3);
  const int vw = orow * REC + lj * CB, vh = orow * REC + 256 + lj * 4, vs = orow * (1024 / G) * 2;
  const int tk = 8 * wave + (lane >> 3), vx = ((t0 + tk) * k + 8 * ((lane & 7) ^ ((tk >> 1) & 7))) * 2;

  ChunkRaw<BITS> rg[2];
  auto issue_w = [&](int sl, ChunkRaw<BITS>& d) __attribute__((always_inline)) {
    sl = sb + (sl < nslab ? sl : nslab - 1);
    const int t = sl >> 4, s16 = sl & 15, tb = t * n * REC;
    if constexpr (BITS == 4) {
      d.w = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, tb + s16 * 32, 0);
    } else {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 lo = __builtin_amdgcn_raw_buffer_load_b64(rw, vw, tb + s16 * 16, 0);
      const uint32_t hi = BITS == 3 ? __builtin_amdgcn_raw_buffer_load_b32(rw, vh, tb + s16 * 8, 0) : 0u;
      d.w = u32x4{lo[0], lo[1], hi, 0u};
    }
    d.s = __builtin_amdgcn_raw_buffer_load_b16(rs, vs, (t * n * (1024 / G) + (G == 128 ? s16 >> 1 : s16)) * 2, 0);
  };
  auto dma_x = [&](int sl, int xs) __attribute__((always_inline)) {
    sl = sb + (sl < nslab ? sl : nslab - 1);
#pragma unroll
    for (int j = 0; j < XPW; ++j)
      lds_dma16(rx, lds + kXBase + xs * kXStage + (wave + NW * j) * 1024, vx + j * 8 * NW * k * 2, sl * kSlab * 2);
  };
  // word u (8 inputs) of the thread's chunk, dequantized into weight stage `stage`
  auto put = [&](const ChunkRaw<BITS>& d, int u, int stage) __attribute__((always_inline)) {
    uint8_t* dst = lds + stage * kWStage + swz(lr, 4 * lj + u);
    const float sc = bf2f(d.s);
    if constexpr (BITS == 4)
      *reinterpret_cast<u32x4*>(dst) = dequant8<OFF>(d.w[u], sc);
    else
      *reinterpret_cast<u32x4*>(dst) = dequant_half<OFF>(half_codes<BITS>(d, u >> 1), sc, u & 1);
  };

  const int wr = (wave % RW) * 64, wtk = (wave / RW) * (T / 2);
  const int l32 = lane & 31, hi = lane >> 5;
  f32x16 acc[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  struct Frag {
    bf16x8 a[2], b[NJ];
  };
  auto frag = [&](int stage, int s, Frag& f) __attribute__((always_inline)) {
    const int q = 2 * s + hi;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      f.a[i] = *reinterpret_cast<const bf16x8*>(lds + stage * kWStage + swz(wr + 32 * i + l32, q));
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      f.b[j] = *reinterpret_cast<const bf16x8*>(lds + kXBase + stage * kXStage + swz(wtk + 32 * j + l32, q));
  };
  auto mfma = [&](const Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
  };
  // the slice's MFMAs and its other instructions in turn: one MFMA, NV VALU
  auto mix = [&](auto NV) __attribute__((always_inline)) {
    static_for<0, 2 * NJ>([&](auto) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_group_barrier(0x0008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x0002, decltype(NV)::value, 0);
    });
    __builtin_amdgcn_sched_barrier(0);
  };

  constexpr int kVmcnt0 = 0x0F70;  // s_waitcnt immediate: vector memory counter 0, the others unconstrained
  constexpr int kVmcntW = kVmcnt0 | kWLoads;  // at most one slab's weight loads outstanding
  Frag f0, f1;
  issue_w(0, rg[0]);
  issue_w(1, rg[1]);
  dma_x(0, 0);
#pragma unroll
  for (int u = 0; u < 4; ++u) put(rg[0], u, 0);
  __builtin_amdgcn_s_waitcnt(kVmcnt0);
  lds_barrier();
  __builtin_amdgcn_sched_barrier(0);
  dma_x(1, 1);
  __builtin_amdgcn_sched_barrier(0);
  issue_w(2, rg[0]);
  __builtin_amdgcn_sched_barrier(0);
  frag(0, 0, f0);
  // slab sl in stage S; f0 holds its first slice.  The order of the token and weight loads is pinned (the counted wait
  // above relies on it); loads past the last slab read it again and are not used
  auto body = [&](int sl, auto S) __attribute__((always_inline)) {
    constexpr int s = decltype(S)::value;
    ChunkRaw<BITS>& d = rg[s ^ 1];  // slab sl + 1
    frag(s, 1, f1);
    mfma(f0);
    put(d, 0, s ^ 1);
    mix(std::integral_constant<int, 4>());
    frag(s, 2, f0);
    mfma(f1);
    put(d, 1, s ^ 1);
    put(d, 2, s ^ 1);
    mix(std::integral_constant<int, 7>());
    frag(s, 3, f1);
    mfma(f0);
    put(d, 3, s ^ 1);
    mix(std::integral_constant<int, 4>());
    // the next slab's token loads have landed (issued a slab ago, before that slab's weight loads)
    __builtin_amdgcn_s_waitcnt(kVmcntW);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    dma_x(sl + 2, s);
    __builtin_amdgcn_sched_barrier(0);
    issue_w(sl + 3, d);
    __builtin_amdgcn_sched_barrier(0);
    frag(s ^ 1, 0, f0);
    mfma(f1);
    __builtin_amdgcn_sched_barrier(0);
  };
  int sl = 0;
  for (; sl + 1 < nslab; sl += 2) {
    body(sl, std::integral_constant<int, 0>());
    body(sl + 1, std::integral_constant<int, 1>());
  }
  if (sl < nslab) body(sl, std::integral_constant<int, 0>());
  __builtin_amdgcn_s_waitcnt(kVmcnt0);  // no load into LDS outlives the workgroup

  // D: register 4 g + e of lane l holds row 8 g + 4 (l / 32) + e of its 32-row tile for token l % 32.  4 rows of a lane's
  // output go in one 8-byte store where the rows stay aligned; else they pass through the wave's share of the LDS, from
  // where the wave writes a token's 64 rows at a time (a lane's own 2-byte stores fall on 32 tokens' rows: 45850 x 1792 W2
  // at 256 tokens 77 us, so 55)
  const bool vec = ((n | ldy) & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0;
  uint8_t* const out = lds + wave * (T * 64);  // [T / 2 tokens][64 rows]: the 8-byte piece c of token t at slot c ^ (t & 15)
  if constexpr (!SPLIT)
    if (!vec) __syncthreads();  // every wave's loads into LDS have landed and its operands are read
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int tk = 32 * j + l32, t = t0 + wtk + tk;
    if (t >= m) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if constexpr (SPLIT) {
          reinterpret_cast<f32x4*>(part)[((size_t)item * (8 * NW * NJ) + ((wave * NJ + j) * 2 + i) * 4 + g) * 64 + lane] =
              f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        } else {
          const int c = 8 * i + 2 * g + hi, r0 = o0 + wr + 4 * c;
          const bf16x2 lo = {(__bf16)acc[i][j][4 * g], (__bf16)acc[i][j][4 * g + 1]};
          const bf16x2 up = {(__bf16)acc[i][j][4 * g + 2], (__bf16)acc[i][j][4 * g + 3]};
          const uint2 v = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, up));
          if (!vec)
            *reinterpret_cast<uint2*>(out + tk * 128 + ((c ^ (tk & 15)) << 3)) = v;
          else if (r0 < n)
            *reinterpret_cast<uint2*>(y + (size_t)t * ldy + r0) = v;
        }
      }
  }
  if constexpr (!SPLIT)
    if (!vec) {
      __syncthreads();
      const int r = o0 + wr + lane, tokens = m - t0 - wtk < T / 2 ? m - t0 - wtk : T / 2;
      if (r < n)
#pragma unroll 8
        for (int tk = 0; tk < tokens; ++tk)
          y[(size_t)(t0 + wtk + tk) * ldy + r] =
              *reinterpret_cast<const uint16_t*>(out + tk * 128 + (((lane >> 2) ^ (tk & 15)) << 3) + 2 * (lane & 3));
    }
}

// y = bf16 of the splits' partials added in order.  A split's partials of a tile lie as its waves hold them (16 bytes per
// lane: 4 rows of one token; R T / 256 such kilobytes per tile), so that they are written and read in whole lines; a
// thread sums one 16-byte piece.  Eight splits' loads are requested before their sums (splits past the last one read the last
// one again and are not added): one memory round trip per eight splits instead of one per split.  A workgroup's four
// kilobytes are 32 rows of 32 tokens: where a lane's 4 outputs are no aligned 8 bytes, they pass through LDS, from where a
// token's 32 rows are written side by side.
__global__ void __launch_bounds__(256) sum_splits_kernel(const f32x4* __restrict__ part, int nsplit, int m, int n,
                                                         uint16_t* __restrict__ y, int ldy, int nrow_tiles, int tiles,
                                                         int R, int nj) {
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;  // kilobyte of the tile, its lane
  const int tile = blockIdx.y, tt = tile / nrow_tiles, rt = tile - tt * nrow_tiles;
  const int wj = f >> 3, wave = wj / nj, j = wj - wave * nj;
  const int rw = R >> 6, wt = wave / rw;  // waves along the rows; the wave along the tokens
  const int tb = (tt * 2 + wt) * 32 * nj + 32 * j, ob = rt * R + (wave - wt * rw) * 64 + 32 * ((f >> 2) & 1);
  const int t = tb + (lane & 31), o = ob + 8 * (f & 3) + 4 * (lane >> 5);
  const bool vec = ((n | ldy) & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0;  // y may be a column offset
  if (vec && (t >= m || o >= n)) return;
  const int kb = R * nj >> 2;  // kilobytes of a tile
  const f32x4* p = part + ((size_t)tile * kb + f) * 64 + lane;
  const size_t step = (size_t)tiles * kb * 64;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < nsplit; s0 += 8) {
    f32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = p[(s0 + i < nsplit ? s0 + i : nsplit - 1) * step];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s0 + i < nsplit) acc += v[i];
  }
  const bf16x2 lo = {(__bf16)acc[0], (__bf16)acc[1]}, hi = {(__bf16)acc[2], (__bf16)acc[3]};
  const uint2 v = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
  if (vec) {
    *reinterpret_cast<uint2*>(y + (size_t)t * ldy + o) = v;
    return;
  }
  __shared__ uint32_t out[32][17];  // [token][32 rows as pairs]
  out[lane & 31][(o - ob) >> 1] = v.x;
  out[lane & 31][((o - ob) >> 1) + 1] = v.y;
  __syncthreads();
  const int r = threadIdx.x & 31;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int tk = (threadIdx.x >> 5) + 8 * q;
    if (tb + tk < m && ob + r < n) y[(size_t)(tb + tk) * ldy + ob + r] = (uint16_t)(out[tk][r >> 1] >> (16 * (r & 1)));
  }
}

template <int BITS, int G, int R, int T, bool SPLIT>
int launch_tiles(const void* x, int m, const void* wt, const void* st, void* y, int n, int ldy, int k, hipStream_t s,
                int nsplit = 1, float* part = nullptr) {
  const int nrt = (n + R - 1) / R, ntt = (m + T - 1) / T;
  const long long grid = ((long long)nrt * ntt * nsplit + 7) / 8 * 8;
  if (grid > 0x7FFFFFFF) return AK_INVALID;
  hipLaunchKernelGGL((wq_gemm_kernel<BITS, G, R, T, SPLIT>), dim3((unsigned)grid), dim3(2 * R),
                     2 * (R + T) * kRowBytes, s, static_cast<const uint16_t*>(x), m,
                     static_cast<const uint8_t*>(wt), static_cast<const uint16_t*>(st), static_cast<uint16_t*>(y), n,
                     ldy, k, nrt, ntt, nsplit, part);
  if (SPLIT)
    hipLaunchKernelGGL(sum_splits_kernel, dim3(R * T / 1024, (unsigned)(nrt * ntt)), dim3(256), 0, s,
                       reinterpret_cast<const f32x4*>(part), nsplit, m, n, static_cast<uint16_t*>(y), ldy, nrt,
                       nrt * ntt, R, T / 64);
  return (int)hipGetLastError();
}

// The tiling of a launch: T tokens per tile and the number of k splits, by the estimated time
//   rounds x (slabs x slab time(R, T) + 3) + (split: 5 + the fp32 partials written and read at 8 TB/s) us,
// rounds = workgroups per XCD / CUs per XCD, rounded up (one workgroup per CU at a time: at T = 64 two fit, but share
// the same throughput).  Slab times measured at 240 workgroups (us): 0.7 at 128 x 128, 0.78 at 256 rows x 64 tokens, 1.12
// at 128, 1.42 at 192, 1.75 at 256 (the dequantization and the weight tile's LDS traffic do not shrink with T).  So wide
// linears take the largest tile that does not pad too many tokens, and narrow or short ones the smallest, with k split
// until one round is nearly full.  Measured
// (us, T x splits): down 5120 x 27648 W2 at 333 tokens 192 x 6 112, 128 x 4 126, 256 x 6 130; at 256 tokens 128 x 6 91,
// 128 x 8 119 (a second round); at 64 tokens 64 x 12 40, 64 x 8 49, 64 x 16 46; o 5120 x 5120 W4 at 256 tokens
// 128 x 6 30, 128 x 4 34, 128 x 8 39.  Splits whose partials exceed kMaxCallScratch (four rounds of 256-token tiles) are
// left out: down at 4096 tokens takes 256 x 3, not 256 x 4.
struct Tiling {
  int R, T, split;
};
long long tiles_of(const Tiling& t, int m, int n) { return (long long)((n + t.R - 1) / t.R) * ((m + t.T - 1) / t.T); }
size_t part_bytes(const Tiling& t, int m, int n) { return (size_t)(tiles_of(t, m, n) * t.split) * 4 * t.R * t.T; }
Tiling pick_tiling(int m, int n, int nslab, bool may_split) {
  const int xcd_cus = num_cus() / 8 > 0 ? num_cus() / 8 : 1;
  Tiling best = {256, 256, 1};
  double best_us = 1e30;
  for (int c = 0; c < 5; ++c) {
    static const struct {
      int R, T;
      double slab;
    } kTiles[5] = {{128, 128, 0.7}, {256, 64, 0.78}, {256, 128, 1.12}, {256, 192, 1.42}, {256, 256, 1.75}};
    for (int sp = 1; sp <= (may_split ? 32 : 1) && (sp == 1 || nslab / sp >= 4); ++sp) {
      const Tiling t = {kTiles[c].R, kTiles[c].T, sp};
      if (sp > 1 && part_bytes(t, m, n) > kMaxCallScratch) break;
      const long long items = tiles_of(t, m, n) * sp, rounds = ((items + 7) / 8 + xcd_cus - 1) / xcd_cus;
      const double us = (double)rounds * ((nslab + sp - 1) / sp * kTiles[c].slab + 3.0) +
                        (sp > 1 ? 5.0 + 2.0 * part_bytes(t, m, n) / 8e6 : 0.0);
      if (us < best_us) best_us = us, best = t;
    }
  }
  return best;
}

template <int BITS, int G, int R, int T>
int launch_t(const void* x, int m, const void* wt, const void* st, void* y, int n, int ldy, int k, hipStream_t s,
             int nsplit, float* part) {
  return part ? launch_tiles<BITS, G, R, T, true>(x, m, wt, st, y, n, ldy, k, s, nsplit, part)
              : launch_tiles<BITS, G, R, T, false>(x, m, wt, st, y, n, ldy, k, s);
}

template <int BITS, int G>
int launch_gemm(const void* x, int m, const void* wt, const void* st, void* y, int n, int ldy, int k, hipStream_t s) {
  // 32-bit buffer offsets: the weights, scales and inputs must each stay below 2 GB
  if ((long long)kpad(k) / 1024 * n * 128 * BITS >= (1ll << 31) || (long long)m * k * 2 >= (1ll << 31))
    return AK_INVALID;
  // fp32 partial tiles of a split launch: in call_scratch; one pass without it (e.g. a capture before any other call)
  Tiling tl = pick_tiling(m, n, k / kSlab, true);
  float* part = nullptr;
  std::unique_lock<std::mutex> lock;
  if (tl.split > 1) {
    lock = std::unique_lock<std::mutex>(scratch_mutex(s));  // the two kernels of a split launch stay together
    part = reinterpret_cast<float*>(call_scratch(s, part_bytes(tl, m, n)).data);
    if (!part) tl = pick_tiling(m, n, k / kSlab, false);
  }
  if (tl.R == 128) return launch_t<BITS, G, 128, 128>(x, m, wt, st, y, n, ldy, k, s, tl.split, part);
  switch (tl.T) {
    case 64: return launch_t<BITS, G, 256, 64>(x, m, wt, st, y, n, ldy, k, s, tl.split, part);
    case 128: return launch_t<BITS, G, 256, 128>(x, m, wt, st, y, n, ldy, k, s, tl.split, part);
    case 192: return launch_t<BITS, G, 256, 192>(x, m, wt, st, y, n, ldy, k, s, tl.split, part);
    default: return launch_t<BITS, G, 256, 256>(x, m, wt, st, y, n, ldy, k, s, tl.split, part);
  }
}

}  // namespace
}  // namespace agq

extern "C" int ak_wq_gemm_tune_query(int m, int n, int k, int* rows, int* tokens, int* splits, size_t* scratch) {
  if (!rows || !tokens || !splits || !scratch || m < 1 || n < 1 || k < 64 || k % 64 != 0) return AK_INVALID;
  const agq::Tiling t = agq::pick_tiling(m, n, k / agq::kSlab, true);
  *rows = t.R, *tokens = t.T, *splits = t.split;
  *scratch = t.split > 1 ? agq::part_bytes(t, m, n) : 0;
  return 0;
}

// No single counterpart in the reference: the fusion of ak_wq_dequant_kt_rows (kernels/src/w4_gemv.cu:877-895) and
// ak_bf16_linear_f32reduce_ld (kernels/src/bf16_linear.cu:68-80), the pair the model's linear() runs above 128 tokens
// (kernels/m1/m1_model.cu:1876-1897).
extern "C" int ak_wq_gemm_kt(int bits, const void* x, int m, const void* wt, const void* st, void* y, int n, int ldy,
                             int k, int group, void* stream) {
  if (!x || !wt || !st || !y || m < 1 || n < 1 || k < 1 || (group != 64 && group != 128) || k % group != 0)
    return AK_INVALID;
  const int ld = ldy ? ldy : n;
  if (ld < n) return AK_INVALID;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  switch (bits * 1000 + group) {
    case 4128: return agq::launch_gemm<4, 128>(x, m, wt, st, y, n, ld, k, s);
    case 4064: return agq::launch_gemm<4, 64>(x, m, wt, st, y, n, ld, k, s);
    case 3128: return agq::launch_gemm<3, 128>(x, m, wt, st, y, n, ld, k, s);
    case 3064: return agq::launch_gemm<3, 64>(x, m, wt, st, y, n, ld, k, s);
    case 2128: return agq::launch_gemm<2, 128>(x, m, wt, st, y, n, ld, k, s);
    case 2064: return agq::launch_gemm<2, 64>(x, m, wt, st, y, n, ld, k, s);
    default: return AK_INVALID;
  }
}
