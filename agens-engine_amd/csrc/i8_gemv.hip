// INT8-weight GEMV for the LM head (W8A16, one fp32 scale per output row), gfx950:
//   y[j][o] (row stride ldy) = bf16(scale[o] * sum_i x[j][i] * q[o][i]),  q int8 [n][k], 1 <= m <= 16, k % 16 == 0.
// Reference: ak_i8_gemv, kernels/src/i8_gemv.cu:28-88.  The reference's numerics are an fp32 order that does not
// depend on m, and this kernel keeps that order exactly, so its results are bit-identical to the reference's:
//   - 32 partial sums per (row, token), partial l over the 16-input chunks c = l, l + 32, l + 64, ... in that order;
//   - per chunk, s = 0 and then s = fma(x_e, q_e, s) for its inputs e = 0..15 in order, and partial += s;
//   - the 32 partials reduced by an xor butterfly (distance 16, 8, 4, 2, 1: v += v[l ^ d]); the result times the
//     row's scale, rounded to bf16 (nearest even).
// Layout on MI355X: a half-wave (32 lanes) plays the reference's warp for kRows rows at once (the lanes' chunk loads
// of a row are 512 contiguous bytes, one 16-byte non-temporal load per lane); the activations' chunk is loaded once
// per token and applied to all of the half-wave's rows (4 for one token, else 2).  A workgroup of 256 threads is 8
// half-waves.  Two to 16 tokens whose activations fit: i8_gemv_lds_kernel below.  The weight stream is
// the only large traffic: at m = 1 the kernel is bounded by HBM (1 byte per weight), from about m = 4 on by the
// VALU (one fma per weight and token).
#include "agens_kernels.h"
#include "wq_common.h"

namespace agq {

int num_cus();

namespace {

// rows per half-wave: 4 for one token (the activation chunk's conversion shared by more rows), 2 with more tokens
// (their accumulators take the registers)
template <int MT>
constexpr int rows_of() { return MT == 1 ? 4 : 2; }

__device__ __forceinline__ float bf_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf_hi(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }
// signed byte B of w as an exact float, one instruction: v_cvt_f32_i32 of the sign-extended byte (SDWA byte select).
// Written out because this toolchain turns (float) of a sign-extended byte into v_cvt_f32_u32 with the same
// sign-extending operand, which converts a negative byte as a large unsigned value.
template <int B>
__device__ __forceinline__ float i8_of(uint32_t w) {
  float r;
  if constexpr (B == 0)
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(r) : "v"(w));
  else if constexpr (B == 1)
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(r) : "v"(w));
  else if constexpr (B == 2)
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(r) : "v"(w));
  else
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(r) : "v"(w));
  return r;
}

// the 16 weights of a chunk word by word as exact floats
__device__ __forceinline__ void chunk_f32(const uint4 q, float (&f)[16]) {
  const uint32_t wd[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[4 * i + 0] = i8_of<0>(wd[i]);
    f[4 * i + 1] = i8_of<1>(wd[i]);
    f[4 * i + 2] = i8_of<2>(wd[i]);
    f[4 * i + 3] = i8_of<3>(wd[i]);
  }
}

// XL: the activations (m * k bf16) staged in LDS by the workgroup, then read from there (one token, k * 2 <= 32 KB)
template <int MT, bool XL>
__global__ void __launch_bounds__(256) i8_gemv_kernel(const uint16_t* __restrict__ x, const int8_t* __restrict__ w,
                                                      const float* __restrict__ scale, uint16_t* __restrict__ y, int m,
                                                      int n, int k, int ldy) {
  constexpr int kRows = rows_of<MT>();
  __shared__ __attribute__((aligned(16))) uint4 xs[XL ? 2048 : 1];
  if constexpr (XL) {
    const uint4* xg = reinterpret_cast<const uint4*>(x);
    for (int i = threadIdx.x; i < (m * k) >> 3; i += 256) xs[i] = xg[i];
    __syncthreads();
  }
  const int l = threadIdx.x & 31;                                          // the reference's lane
  const int hw = threadIdx.x >> 5;                                         // half-wave of the workgroup
  const int o0 = (blockIdx.x * (256 / 32) + hw) * kRows;                   // first row of this half-wave
  const int chunks = k >> 4;
  float acc[kRows][MT];
#pragma unroll
  for (int r = 0; r < kRows; ++r)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[r][j] = 0.f;
  // rows past n read row n - 1 (results not written)
  const int8_t* wr[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) wr[r] = w + (size_t)(o0 + r < n ? o0 + r : n - 1) * k;
  // the next chunk's weights are requested before this chunk is computed (two chunks in flight per row); the two
  // half-waves of a wave read different rows: per-lane addresses
  u32x4 nx[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r)
    nx[r] = l < chunks ? __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wr[r] + (size_t)l * 16))
                       : u32x4{0u, 0u, 0u, 0u};
  for (int c = l; c < chunks; c += 32) {
    float qf[kRows][16];
    u32x4 cur[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) cur[r] = nx[r];
    if (c + 32 < chunks) {
#pragma unroll
      for (int r = 0; r < kRows; ++r)
        nx[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wr[r] + (size_t)(c + 32) * 16));
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) chunk_f32(make_uint4(cur[r][0], cur[r][1], cur[r][2], cur[r][3]), qf[r]);
    // tokens: every j < MT unrolled (a guard, not a loop exit, so that the accumulators stay in registers)
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      if (j < m) {
        const uint4* xr = (XL ? xs : reinterpret_cast<const uint4*>(x)) + (((size_t)j * k) >> 3) + 2 * c;
        const uint4 a = xr[0], b = xr[1];
        const uint32_t xw[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        float xf[16];
#pragma unroll
        for (int i = 0; i < 8; ++i) xf[2 * i] = bf_lo(xw[i]), xf[2 * i + 1] = bf_hi(xw[i]);
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
          float s = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e) s = __builtin_fmaf(xf[e], qf[r][e], s);
          acc[r][j] += s;
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const int o = o0 + r;
    const float sc = o < n ? scale[o] : 0.f;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      if (j < m) {
        float v = acc[r][j];
#pragma unroll
        for (int d = 16; d > 0; d >>= 1) v += __shfl_xor(v, d, 32);
        if (l == 0 && o < n) y[(size_t)j * ldy + o] = f2bf(v * sc);
      }
    }
  }
}

constexpr int kRsrcWord3 = 0x00020000;  // raw buffer resource, dword 3 (CDNA)

// The same sums for MT tokens with their activations in LDS: persistent workgroups that take groups of 8 R rows (R per
// half-wave) in turn.  With the activations read from memory, every token's chunk was waited for in order behind the
// next weights, which drained the weight stream once per chunk; here the next chunk's weights (of the next group at a
// group's end) are the only loads outstanding, and they stay in flight over a whole chunk.  A token's chunk is read from
// LDS while the chains of the token before run (two planes of 16-byte halves: no bank conflicts) and is unpacked once
// for R rows.  What is left is the VALU: per weight MT fmas (the reference's order), one conversion and MT / R unpacking
// operations; at 4 tokens and R = 4 about 125 us of the 148 measured for 152064 x 5120, at 8 tokens nearly
// all of the 228.
template <int MT, int R>
__global__ void __launch_bounds__(256, R == 4 ? 3 : 4) i8_gemv_lds_kernel(
    const uint16_t* __restrict__ x, const int8_t* __restrict__ w, const float* __restrict__ scale,
    uint16_t* __restrict__ y, int n, int k, int ldy) {
  constexpr int NV = R * MT, GR = 8 * R;
  extern __shared__ __attribute__((aligned(16))) u32x4 xs[];  // [token][chunk half][chunk]
  const int chunks = k >> 4;
  for (int i = threadIdx.x; i < MT * chunks * 2; i += 256) {
    const int t = i / (2 * chunks), p = i - t * 2 * chunks;
    xs[(t * 2 + (p & 1)) * chunks + (p >> 1)] = reinterpret_cast<const u32x4*>(x)[i];
  }
  __syncthreads();
  const int l = threadIdx.x & 31, hw = threadIdx.x >> 5;
  const int groups = (n + GR - 1) / GR, iters = (chunks + 31) >> 5;
  auto rows_of_group = [&](int g) __attribute__((always_inline)) {
    const int g1 = g < groups ? g : (int)blockIdx.x;  // past the end: the first group again, not used
    const int nr = n - g1 * GR < GR ? n - g1 * GR : GR;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(w + (size_t)g1 * GR * k), (short)0, nr * k, kRsrcWord3);
  };
  const int vo = hw * R * k + l * 16;
  u32x4 nx[R];
  auto fetch = [&](int g, int it) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rw = rows_of_group(g);
#pragma unroll
    for (int r = 0; r < R; ++r) nx[r] = __builtin_amdgcn_raw_buffer_load_b128(rw, vo + r * k + it * 512, 0, 2);
  };
  // the value (row idx % R, token idx / R) that this lane ends with (the reduction below), and whether it writes it
  constexpr int NP = NV <= 2 ? 2 : NV <= 4 ? 4 : NV <= 8 ? 8 : NV <= 16 ? 16 : 32;  // values padded to a power of two
  int idx = 0;
#pragma unroll
  for (int st = 0; st < 5; ++st) idx += l & (16 >> st) ? NP >> st >> 1 : 0;
  const bool wr = idx < NV && (l & (32 / NP - 1)) == 0;
  fetch(blockIdx.x, 0);
  for (int g = blockIdx.x; g < groups; g += gridDim.x) {
    const int o = g * GR + hw * R + idx % R;
    const float sc = scale[o < n ? o : n - 1];
    float acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.f;
    for (int it = 0; it < iters; ++it) {
      float qf[R][16];
#pragma unroll
      for (int r = 0; r < R; ++r) chunk_f32(make_uint4(nx[r][0], nx[r][1], nx[r][2], nx[r][3]), qf[r]);
      const bool last = it + 1 == iters;
      fetch(last ? g + (int)gridDim.x : g, last ? 0 : it + 1);
      const int c = it * 32 + l;
      if (c < chunks) {
        // the next token's chunk is read while this one's chains run
        u32x4 a = xs[c], b = xs[chunks + c];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          const u32x4 ca = a, cb = b;
          if (j + 1 < MT) a = xs[(2 * j + 2) * chunks + c], b = xs[(2 * j + 3) * chunks + c];
          float xf[16];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            xf[2 * i] = bf_lo(ca[i]), xf[2 * i + 1] = bf_hi(ca[i]);
            xf[8 + 2 * i] = bf_lo(cb[i]), xf[9 + 2 * i] = bf_hi(cb[i]);
          }
          float s[R];
#pragma unroll
          for (int r = 0; r < R; ++r) s[r] = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e)
#pragma unroll
            for (int r = 0; r < R; ++r) s[r] = __builtin_fmaf(xf[e], qf[r][e], s[r]);
#pragma unroll
          for (int r = 0; r < R; ++r) acc[j * R + r] += s[r];
        }
      }
    }
    // the butterfly over the 32 lanes, each step exchanging the half of the values that the partner keeps (both lanes of
    // a pair would form the same sum): lane l ends with the values of the index bits its lane bits stand for
#pragma unroll
    for (int st = 0; st < 5; ++st) {
      const int d = 16 >> st, cnt = NP >> st >> 1;  // values left after this step
      if (cnt >= 1) {
        const bool up = l & d;
#pragma unroll
        for (int i = 0; i < cnt; ++i) {
          const float lo = i < NV ? acc[i] : 0.f, hi = i + cnt < NV ? acc[i + cnt < NV ? i + cnt : 0] : 0.f;
          acc[i < NV ? i : 0] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, d, 32);
        }
      } else {
        acc[0] += __shfl_xor(acc[0], d, 32);
      }
    }
    if (o < n && wr) y[(size_t)(idx / R) * ldy + o] = f2bf(acc[0] * sc);
  }
}

template <int MT, int R>
void launch_lds(const uint16_t* x, const int8_t* w, const float* scale, uint16_t* y, int n, int k, int ldy,
                hipStream_t s) {
  // as many workgroups per CU as the LDS and the registers (3 of 4 rows, 4 of 2 rows per half-wave) take
  const size_t smem = (size_t)MT * k * 2, fit = (size_t)160 * 1024 / smem;
  const int per = fit < (R == 4 ? 3 : 4) ? (int)fit : (R == 4 ? 3 : 4);
  const int groups = (n + 8 * R - 1) / (8 * R), grid = groups < num_cus() * per ? groups : num_cus() * per;
  hipLaunchKernelGGL((i8_gemv_lds_kernel<MT, R>), dim3(grid), dim3(256), smem, s, x, w, scale, y, n, k, ldy);
}

template <int MT>
void launch_lds_rows(const uint16_t* x, const int8_t* w, const float* scale, uint16_t* y, int n, int k, int ldy,
                     hipStream_t s) {
  // 2 rows per half-wave where 4 leave CUs idle (8001 x 1040, 8 tokens 8.2 against 9.2 us; 20000 x 2000 18.7 / 19.5;
  // 152064 x 5120 274 / 233)
  if (n < 32768)
    launch_lds<MT, 2>(x, w, scale, y, n, k, ldy, s);
  else
    launch_lds<MT, 4>(x, w, scale, y, n, k, ldy, s);
}

void lds_part(const uint16_t* x, const int8_t* w, const float* scale, uint16_t* y, int m, int n, int k, int ldy,
              hipStream_t s) {
  switch (m) {
    case 2: return launch_lds_rows<2>(x, w, scale, y, n, k, ldy, s);
    case 3: return launch_lds_rows<3>(x, w, scale, y, n, k, ldy, s);
    case 4: return launch_lds_rows<4>(x, w, scale, y, n, k, ldy, s);
    case 5: return launch_lds_rows<5>(x, w, scale, y, n, k, ldy, s);
    case 6: return launch_lds_rows<6>(x, w, scale, y, n, k, ldy, s);
    case 7: return launch_lds_rows<7>(x, w, scale, y, n, k, ldy, s);
    default: return launch_lds_rows<8>(x, w, scale, y, n, k, ldy, s);
  }
}

}  // namespace
}  // namespace agq

extern "C" int ak_i8_gemv(const void* x, const void* w, const void* scale, void* y, int m, int n, int k, int ldy,
                          void* stream) {
  // the reference's checks (i8_gemv.cu:74), and null pointers / empty shapes
  if (!x || !w || !scale || !y || m < 1 || m > 16 || n < 1 || k < 16 || k % 16) return AK_INVALID;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto X = static_cast<const uint16_t*>(x);
  auto W = static_cast<const int8_t*>(w);
  auto S = static_cast<const float*>(scale);
  auto Y = static_cast<uint16_t*>(y);
  auto wgs = [n](int rows) { return dim3((n + 8 * rows - 1) / (8 * rows)); };  // 8 half-waves per workgroup
  // Two to 16 tokens in parts of at most 8 whose activations take at most 80 KB of LDS (two workgroups per CU): the LDS
  // kernel where one part covers them, or two.  Measured (us, 152064 x 5120, before = activations from L1 per token and
  // row pair): 2 / 4 / 8 / 16 tokens 156 / 233 / 358 / 628 -> 119 / 148 / 228 / 460.  Two or three tokens on less than 32
  // MB of weights stay with the kernel below (8001 x 1040: 7.1 against 7.4, 7.4 against 7.7).
  // The second part reads all weights again.  Below 80 MB the caches still hold most of them, and four tokens or more gain
  // (1700 x 20480, 4 tokens 61.8 -> 53.8; 6000 x 13648, 6 tokens 64.8 -> 49.9; but 6000 x 16400, 94 MB, 4 tokens 52.7 ->
  // 54.9); above, it pays only for parts of up to four tokens or more (60000 x 10240, 8 tokens 294 -> 267; 33000 x 8192, 9
  // tokens 176 -> 136), not for less (12000 x 24576, 2 tokens 73 against 104; 12000 x 16400, 4 tokens 78 against 97; 60000
  // x 12288, 6 tokens 319 against 338).
  const int cap = 40960 / k, most = cap < 8 ? cap : 8;
  const long long bytes = (long long)n * k;
  const bool one = m > 1 && m <= most && (m > 3 || bytes >= 32 << 20);
  const bool two = m > 3 && m > most && m <= 2 * most && (most >= 4 || bytes < 80 << 20);
  if (one || two) {
    const int parts = (m + most - 1) / most, per = (m + parts - 1) / parts;
    for (int m0 = 0; m0 < m; m0 += per)
      agq::lds_part(X + (size_t)m0 * k, W, S, Y + (size_t)m0 * ldy, m - m0 < per ? m - m0 : per, n, k, ldy, s);
    return (int)hipGetLastError();
  }
  if (m == 1 && k <= 16384)
    hipLaunchKernelGGL((agq::i8_gemv_kernel<1, true>), wgs(agq::rows_of<1>()), dim3(256), 0, s, X, W, S, Y, m, n, k,
                       ldy);
  else if (m == 1)
    hipLaunchKernelGGL((agq::i8_gemv_kernel<1, false>), wgs(agq::rows_of<1>()), dim3(256), 0, s, X, W, S, Y, m, n, k,
                       ldy);
  else if (m <= 8)
    hipLaunchKernelGGL((agq::i8_gemv_kernel<8, false>), wgs(agq::rows_of<8>()), dim3(256), 0, s, X, W, S, Y, m, n, k,
                       ldy);
  else
    hipLaunchKernelGGL((agq::i8_gemv_kernel<16, false>), wgs(agq::rows_of<16>()), dim3(256), 0, s, X, W, S, Y, m, n,
                       k, ldy);
  return (int)hipGetLastError();
}
