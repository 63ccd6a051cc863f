// Batch-invariant bf16 GEMV for small m (speculative decoding: a verify of m tokens must give every token the bits a
// one-token step gives it), gfx950:
//   y[t][r] (row stride ldy) = bf16(sum_i x[t][i] * W[r][i] (+ bias[r])),  W bf16 [n][k] row-major, 1 <= m <= 128,
//   k % 32 == 0.
// Reference: ak_bf16_gemv_bi / _ld, kernels/src/bi_gemv.cu:270-356 (tensor-core MMA kernels whose per-token order is the
// same for every m).  The reference's bits come from its MMA instruction's internal accumulation, which no other
// hardware reproduces; this kernel keeps the reference's contract instead -- fp32 accumulation, the bias added in fp32
// before the one bf16 rounding, and an order that does not depend on m:
//   - k is cut into 64-input steps and those into 8 contiguous chunks, chunk p = steps [p S / 8, (p + 1) S / 8) of S;
//     wave p of a workgroup takes chunk p for the workgroup's 16 RB rows, each step two v_mfma_f32_16x16x32_bf16 (inputs
//     [64 s, 64 s + 32) then [64 s + 32, 64 s + 64)) accumulating in fp32;
//   - the MFMA's A operand is 16 weight rows, its B operand 16 tokens: the columns of the result are independent, so a
//     token's sums do not depend on the other tokens; more than 16 tokens are more B tiles of the same steps;
//   - the 8 chunks' partial sums are added in order (from chunk 0), then the bias, then the bf16 rounding.
// Operands: lane (c, h) = (l % 16, l / 16) holds inputs 8 h .. + 8 of row (A) / token (B) c of the 32-input slice; any
// input-to-slot map gives the same sum as long as A and B use the same one.  D: lane (c, h) holds rows 4 h + i, i < 4, of
// token c.
// What bounds it: at few tokens the HBM stream and the latency of a short chain (5120 x 5120: 10 steps per wave), at
// more the activations, which every workgroup reads whole from L2.  So every load instruction reads whole 128-byte
// lines of 8 rows (or tokens): the lanes of a pair load the two halves of one row's line and swap them by DPP (own_row);
// the next KU steps are requested before these are used; rows past n, tokens past m and steps past a chunk read zeros
// through the buffers' range, which costs no memory traffic; and a workgroup takes 32 rows where that saves a round of
// workgroups or activation traffic (rows_per_workgroup).  Measured (us, before = half-line loads at clamped addresses,
// one row block per workgroup): 5120 x 5120 at 1 / 16 / 64 / 128 tokens 20.4 / 28.6 / 54.7 / 89.9 -> 13.2 / 15.8 / 27.5 /
// 40.4; 8000 x 8192 at 4 tokens 35.0 -> 22.0 (5.95 TB/s).  16 waves per workgroup were slower (5120 x 5120 at 1 token
// 18.5), and so were 3 or 4 steps per request group (19.7, 18.0 at 16 tokens).
#include "agens_kernels.h"
#include "wq_common.h"

#include <algorithm>

namespace agq {

int num_cus();

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int NW = 8;  // waves per workgroup, chunks of k
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer resource, dword 3 (CDNA)

// a = load 0, b = load 1 of a lane pair (lanes 2 i, 2 i + 1: row 2 i, then row 2 i + 1; the even lane the first half of
// the line, the odd lane the second) -> the first and second half of the lane's own row
__device__ __forceinline__ void own_row(u32x4& a, u32x4& b, bool odd) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t v = odd ? a[i] : b[i];  // what the partner lane needs
    const uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);  // quad_perm [1, 0, 3, 2]
    a[i] = odd ? r : a[i];
    b[i] = odd ? b[i] : r;
  }
}

// TT token tiles of 16 (m <= 16 TT), RB row blocks of 16 per workgroup, KU steps per group of requests.  WIDE: rows of
// 2^24 inputs or more, which the buffers' 32-bit offsets do not cover: the same loads by address, at clamped rows, tokens
// and inputs in place of zeros (what they hold is not used)
template <int TT, int RB, int KU, bool WIDE = false>
__global__ void __launch_bounds__(NW * 64) bi_gemv_kernel(const uint16_t* __restrict__ x, int m,
                                                              const uint16_t* __restrict__ w,
                                                              const uint16_t* __restrict__ bias,
                                                              uint16_t* __restrict__ y, int n, int k, long ldy) {
  extern __shared__ f32x4 red[];  // [NW][RB * TT][64]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, h = lane >> 4;
  const bool odd = c & 1;
  const int row0 = (int)blockIdx.x * 16 * RB;
  const int steps = (int)(((unsigned)k + 63) >> 6), s_lo = wave * steps / NW, s_hi = (wave + 1) * steps / NW;
  // bytes of a lane's two loads within a step: the half line (c & 1), chunk h of it
  const unsigned lo = 64 * (c & 1) + 16 * h, k2 = 2u * k;
  const int nr = n - row0 < 16 * RB ? n - row0 : 16 * RB;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w + (size_t)row0 * k),
                                                                      (short)0, (int)(nr * k2), kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), (short)0, (int)(m * k2),
                                                                      kRsrcWord3);
  const unsigned v0 = (c & ~1) * k2 + lo;  // the lane's first load: row (token) c & ~1 of a block; the second a row further
  f32x4 acc[RB][TT];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Step {
    u32x4 a[RB][2], b[TT][2];
  };
  // a step's loads; rows past n and tokens past m read zeros (out of the buffers' range), steps past the wave's last
  // are not used and mostly out of range too
  auto load = [&](int s, Step& d) __attribute__((always_inline)) {
    if constexpr (WIDE) {
      const int i = s < s_hi ? 64 * s + 32 * (c & 1) + 8 * h : 0, i1 = (unsigned)i < (unsigned)k ? i : 0;
      auto at = [&](const uint16_t* p, int r, int rows) {
        return __builtin_nontemporal_load(
            reinterpret_cast<const u32x4*>(p + (size_t)(r < rows ? r : rows - 1) * k + i1));
      };
#pragma unroll
      for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int r = 0; r < RB; ++r) d.a[r][e] = at(w, row0 + 16 * r + (c & ~1) + e, n);
#pragma unroll
        for (int t = 0; t < TT; ++t) d.b[t][e] = at(x, 16 * t + (c & ~1) + e, m);
      }
      return;
    }
    const unsigned v = v0 + (s < s_hi ? 128u * s : 0x40000000u);
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int e = 0; e < 2; ++e) d.a[r][e] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(v + (16 * r + e) * k2), 0, 2);
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e) d.b[t][e] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(v + (16 * t + e) * k2), 0, 0);
  };
  auto use = [&](int s, Step& d) __attribute__((always_inline)) {
    if (s >= s_hi) return;
    const bool cut = 64u * s + 32 >= (unsigned)k;
    const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      own_row(d.a[r][0], d.a[r][1], odd);
      if (cut) d.a[r][1] = z;
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      own_row(d.b[t][0], d.b[t][1], odd);
      if (cut) d.b[t][1] = z;
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int r = 0; r < RB; ++r)
          acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, d.a[r][e]),
                                                              __builtin_bit_cast(bf16x8, d.b[t][e]), acc[r][t], 0, 0, 0);
  };
  if (s_lo < s_hi) {
    // two groups of steps in turn, the next one requested before this one is used (no request past the last step: a
    // branch around the loads alone would make their wait counts conservative, so the last use is a path of its own)
    Step st[2][KU];
    auto load_group = [&](int s, Step (&d)[KU]) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < KU; ++u) load(s + u, d[u]);
    };
    auto use_group = [&](int s, Step (&d)[KU]) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < KU; ++u) use(s + u, d[u]);
    };
    load_group(s_lo, st[0]);
    if constexpr (TT * RB >= 8) {  // registers for one copy of the uses only: the last requests are past the chunk
      for (int s = s_lo; s < s_hi; s += 2 * KU) {
        load_group(s + KU, st[1]);
        use_group(s, st[0]);
        load_group(s + 2 * KU, st[0]);
        use_group(s + KU, st[1]);
      }
    } else for (int s = s_lo;; s += 2 * KU) {
      if (s + KU >= s_hi) {
        use_group(s, st[0]);
        break;
      }
      load_group(s + KU, st[1]);
      use_group(s, st[0]);
      if (s + 2 * KU >= s_hi) {
        use_group(s + KU, st[1]);
        break;
      }
      load_group(s + 2 * KU, st[0]);
      use_group(s + KU, st[1]);
    }
  }
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t) red[(wave * RB * TT + r * TT + t) * 64 + lane] = acc[r][t];
  __syncthreads();
  // wave i adds the chunks' partials of tiles i, i + 8, .. in chunk order, then the bias, and writes 4 rows of a token
  for (int i = wave; i < RB * TT; i += NW) {
    const int r = i / TT, t = i - r * TT;
    f32x4 v = red[i * 64 + lane];
#pragma unroll
    for (int ww = 1; ww < NW; ++ww) v += red[(ww * RB * TT + i) * 64 + lane];
    const int tok = 16 * t + c;
    if (tok < m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = row0 + 16 * r + 4 * h + e;
        if (row < n) {
          const float b = bias ? __uint_as_float((uint32_t)bias[row] << 16) : 0.f;
          y[(size_t)tok * ldy + row] = f2bf(bias ? v[e] + b : v[e]);
        }
      }
    }
  }
}

template <int TT, int RB, int KU, bool WIDE = false>
void launch_bi(const uint16_t* x, int m, const uint16_t* w, const uint16_t* bias, uint16_t* y, int n, int k, long ldy,
               hipStream_t s) {
  hipLaunchKernelGGL((bi_gemv_kernel<TT, RB, KU, WIDE>), dim3((n + 16 * RB - 1) / (16 * RB)), dim3(NW * 64),
                     NW * RB * TT * 64 * sizeof(f32x4), s, x, m, w, bias, y, n, k, ldy);
}

// Row blocks per workgroup, 1 or 2 (the same results).  Workgroups take rounds of one per CU (two on a CU share its
// throughput); a round of one-block workgroups takes u, of two-block ones r u, unless the weights' stream is longer,
// which runs faster with more workgroups (7.3 against 6.0 TB/s).  Measured at k = 5120 (us, one / two blocks): 16 tokens
// n = 4096 11.5 / 15.7, 5120 19.1 / 15.9, 8192 20.1 / 17.2, 12000 27.7 / 29.2; 1 token n = 20000 33.8 / 36.4; 64 tokens n
// = 3200 20.8 / 26.6, 4500 36.1 / 26.1; k = 8192, 4 tokens n = 8000 22.0 / 26.9.
int rows_per_workgroup(int n, int k, int m) {
  const double u = (m <= 16 ? 5.0 + 2.5 * m / 16 : m <= 32 ? 11.0 : m <= 64 ? 16.5 : 29.0) * k / 5120;
  const double r = m <= 16 ? 1.5 : m <= 32 ? 1.4 : m <= 64 ? 1.33 : 1.2, bytes = 2.0 * n * k;
  const int nb = (n + 15) / 16, cus = num_cus();
  const double one = (nb + cus - 1) / cus * u, two = (nb + 2 * cus - 1) / (2 * cus) * r * u;
  return std::max(two, bytes / 6.0e6) < std::max(one, bytes / 7.3e6) ? 2 : 1;
}

template <int TT, int KU1, int KU2>
void launch_rows(const uint16_t* x, int m, const uint16_t* w, const uint16_t* bias, uint16_t* y, int n, int k, long ldy,
                 hipStream_t s) {
  if (k >= 1 << 24)  // (128 tokens or 32 rows of fewer inputs stay within 32-bit buffer offsets)
    launch_bi<TT, 1, KU1, true>(x, m, w, bias, y, n, k, ldy, s);
  else if (rows_per_workgroup(n, k, m) == 2)
    launch_bi<TT, 2, KU2>(x, m, w, bias, y, n, k, ldy, s);
  else
    launch_bi<TT, 1, KU1>(x, m, w, bias, y, n, k, ldy, s);
}

}  // namespace
}  // namespace agq

extern "C" int ak_bf16_gemv_bi_ld(const void* x, const void* w, const void* bias, void* y, int m, int n, int k, long ldy,
                                  void* stream) {
  // the reference's checks (bi_gemv.cu:276), null pointers / empty shapes, and a row stride below n (token rows would
  // overlap)
  if (!x || !w || !y || m < 1 || m > 128 || n < 1 || k < 32 || k % 32 != 0 || ldy < n) return AK_INVALID;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto X = static_cast<const uint16_t*>(x);
  auto W = static_cast<const uint16_t*>(w);
  auto B = static_cast<const uint16_t*>(bias);
  auto Y = static_cast<uint16_t*>(y);
  switch ((m + 15) / 16) {
    case 1: agq::launch_rows<1, 2, 2>(X, m, W, B, Y, n, k, ldy, s); break;
    case 2: agq::launch_rows<2, 2, 2>(X, m, W, B, Y, n, k, ldy, s); break;
    case 3:
    case 4: agq::launch_rows<4, 1, 1>(X, m, W, B, Y, n, k, ldy, s); break;
    default: agq::launch_rows<8, 1, 1>(X, m, W, B, Y, n, k, ldy, s); break;
  }
  return (int)hipGetLastError();
}

extern "C" int ak_bf16_gemv_bi(const void* x, const void* w, const void* bias, void* y, int m, int n, int k,
                               void* stream) {
  return ak_bf16_gemv_bi_ld(x, w, bias, y, m, n, k, n, stream);
}
