// GEMV entry points of the C ABI: argument rules, routing between the two numerics and token chunking.  Split-K
// launches keep stripe partials and row-range counters in library scratch, the tiled kernel its converted activations as
// well (wq_scratch.h: without scratch, e.g. in a capture before any other call, a route that needs none is taken), or,
// for ak_wq_gemv_kt_multi_noalloc, in a static device array; every other launch is self-contained (partials meet in LDS).
//
// Argument rules and return codes follow the reference (kernels/src/w4_gemv.cu:702-731, :852-876, :898-935,
// :3265-3282): group in {64, 128} with k % group == 0, 1 <= nseg <= 4, 1 <= m <= 128; error 1 otherwise.
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <new>

#include "agens_kernels.h"
#include "agens_tuning.h"
#include "wq_common.h"

namespace agq {

int exact_gemv(int bits, const void* x, int m, const Segs& g, int k, int group, int bf16w, hipStream_t s);
int exact_ct_gemv(const void* x, const int32_t* packed, const void* scales, void* y, int n, int k, hipStream_t s);
int i8_gemv(int bits, const void* x, int m, const Segs& g, int k, int group, hipStream_t s);
int i8_gemv_m1(int bits, const void* x, int m, const Segs& g, int k, int group, hipStream_t s, int act = 0);
int i8_gemv_mt(int bits, const void* x, int m, const Segs& g, int k, int group, hipStream_t s, int act = 0);
int tile_gemv(int bits, const void* x, int m, const Segs& g, int k, int group, hipStream_t s, int act);
int mm_gemv(int bits, const void* x, int m, const Segs& g, int k, int group, hipStream_t s, int act);
int num_cus();
int m1d_chain_make(int nsteps, const int* bits, const void* const* x, const int* m, const int* k, const Segs* segs,
                   const int* wait, const int* act, void** table, int* mt_out, size_t* smem_out);
int m1d_chain_launch(const void* table, int nsteps, int mt, size_t smem, hipStream_t s);
int mt_chain_make(int nsteps, const int* bits, const void* const* x, const int* m, const int* k, const Segs* segs,
                  const int* wait, void** table, int* nt_out, size_t* smem_out);
int mt_chain_launch(const void* table, int nsteps, int nt, size_t smem, hipStream_t s);
int mt_chain_error(int* err);
int m1d_chain_error(int* err);
void m1d_tune_override(int split, int nwv, int sk);
int m1d_tune_query(int bits, int m, const Segs& g, int k, int* split, int* nwv, int* sk);

namespace {

constexpr int kMaxTokensPerLaunch = 16;

// Process-global switches (tuning and test selections, not per-call state): atomics, so that a switch set on one
// thread while another launches is read whole; a launch sees the value set before it or after it.
std::atomic<int> g_mode{-1};  // -1: environment (AGENS_W4_EXACT=1 selects the exact path), 0: exact, 1: integer MFMA

bool exact_mode() {
  const int mode = g_mode.load(std::memory_order_relaxed);
  if (mode >= 0) return mode == 0;
  static int env = -1;
  if (env < 0) {
    const char* v = getenv("AGENS_W4_EXACT");
    env = (v && v[0] == '1') ? 1 : 0;
  }
  return env == 1;
}

// The smallest token count routed to the fp16-MFMA kernel (wq_mm.hip) in the default numerics, where the tiled kernel
// (tile_route) does not take the call: the measured crossover with the integer-limb kernels (below it those are faster).
// Both compute the same numerics bit for bit, so the switch changes speed only.  0: never; set through ak_wq_set_mm_min
// or AGENS_WQ_MM_MIN.  Above kMmMaxK inputs the integer kernels stay faster at every token count (measured: down 5120 x
// 27648 at 24..128 tokens).
constexpr int kMmMinDefault = 17;
constexpr int kMmMaxK = 8192;
std::atomic<int> g_mm_min{-1};

// the explicit crossover (ak_wq_set_mm_min, else AGENS_WQ_MM_MIN), or -1 for the compiled-in rule
int mm_min_set() {
  const int v = g_mm_min.load(std::memory_order_relaxed);
  if (v >= 0) return v;
  static int env = -2;
  if (env == -2) {
    const char* e = getenv("AGENS_WQ_MM_MIN");
    env = e && e[0] ? atoi(e) : -1;
  }
  return env;
}

// whether a default-numerics call of m tokens takes the fp16-MFMA kernel (the kernel itself takes group 128 only): an
// explicit crossover applies at every k, the compiled-in one up to kMmMaxK inputs
bool mm_route(int m, int k, int group, bool exact) {
  if (exact || group != 128) return false;
  const int set = mm_min_set();
  if (set >= 0) return set > 0 && m >= set;
  return m >= kMmMinDefault && k <= kMmMaxK;
}

// Group 64 at one and two tokens: whether the any-m kernel (wq_i8.hip) is the faster one.  Its workgroups own 64 rows and
// all inputs, a wave per stripe, two workgroups per CU: a round of them takes about as long however full it is, and up to
// 8 tiles of 1024 inputs hardly longer for more inputs.  The tiled kernel's time is proportional to both.  So the line is
// where a round (or its half with one workgroup per CU) is well filled.  Measured (us, any-m / tiled, 1 token):
//   second half of a round: 32768 x 8192 W4 42 / 58, 29000 x 5120 34 / 37, 23500 x 6144 W2 35 / 38, but 21000 x 6144 37 /
//     31, 23500 x 5120 33 / 30; 2 tokens 32768 x 8192 W4 44 / 58, 26000 x 8192 44 / 46, 21000 x 8192 43 / 42;
//   9 tiles and more (two tiles per wave: the any-m kernel's step up): 32768 x 10240 W2 59 / 68, 17500 x 9216 52 / 58, but
//     17500 x 12288 60 / 55; 2 tokens 26000 x 10240 96 / 66 (one workgroup per CU: the activations' LDS);
//   first half: 15000 x 5120 W4 27 / 29, W3 33 / 35, W2 26 / 26, 11000 x 5120 W4 26 / 22;
//   third round, from its first half on: 98304 x 8192 W4 117 / 130, 82000 x 8192 110 / 124; the tiled kernel at 57000,
//     65536 and 115000 rows (78 / 75, 80 / 78, 148 / 131).
bool any_m_route(int bits, int m, const Segs& g, int k) {
  if (m > 2) return false;
  const int cus = num_cus(), wg = (g.end[g.nseg - 1] + 63) / 64, tiles = kpad(k) / 1024;
  if (wg <= cus) return m == 1 && bits >= 3 && tiles >= 5 && tiles <= 6 && wg >= 4 * cus / 5;
  if (wg <= 2 * cus) {
    if (tiles <= 8) return tiles >= 5 && (long long)2 * wg * tiles >= 17 * cus && (m == 1 || 2 * wg >= 3 * cus);
    return m == 1 && tiles <= 14 && wg >= cus + cus / 8 * (tiles - 9);
  }
  return m == 1 && tiles >= 7 && tiles <= 8 && wg > 4 * cus && wg <= 6 * cus;
}

// Whether a default-numerics call takes the tiled kernel (wq_tile.hip; same bits).  An explicit crossover keeps the older
// kernels.  Measured, the older kernels' time -> the tiled kernel's, us:
//   group 64 (which the small-M kernels do not take), every token count but for any_m_route: 5120 x 6144 W4 28 -> 18 at 1
//     token, 188 -> 19 at 16; 55296 x 5120 W3 84 -> 66 and 624 -> 70; 152064 x 5120 W4 153 -> 127 at 1; 64 x 64 14.8 -> 11.1;
//   group 128 from 33 tokens: 55296 x 5120 W3 164 -> 86 at 64 tokens, 5120 x 5120 W4 38.6 -> 28.9, 5120 x 27648 W3 130 ->
//     68, 64 x 512 19.8 -> 12.3; at 17 to 32 tokens on wide linears, 55296 x 5120 W3 82 -> 60, 14000 x 2560 W3 29.4 -> 22,
//     7168 x 5120 W4 25.9 -> 24.2 at 17, but 5120 x 5120 W4 19.7 -> 20.4 and 1000 x 2048 W3 12.5 -> 13.6: the fp16-MFMA
//     kernel up to kTileRows rows, at 3 tiles of inputs up to its one round of 8192 (kTileRows3: 6200 x 3072 W2 at 32
//     tokens 15.8 -> 17.4, 7680 x 3072 W3 17.3 -> 18.2, 8208 x 3072 27.0 -> 17.7; 4 tiles 6200 rows 17.5 -> 18.1, 8192
//     rows the same; 2 tiles 0.97); past kMmMaxK inputs, where the other side is the integer kernels in chunks of 16
//     tokens, from 24: 5120 x 27648 W2 51.9 -> 47.4 at 24, 45.5 -> 47.3 at 20;
//     and not where tile_gemv leaves 33 to 40 tokens of long k to the integer kernels (integer_kernels_faster);
//   up to 16 tokens at group 128 the small-M kernels (55296 x 5120 W3, 16 tokens: 46 against 49).
constexpr int kTileRows = 6144, kTileRows3 = 8192;
bool tile_route(int bits, int m, const Segs& g, int k, int group, bool exact) {
  if (exact || mm_min_set() >= 0) return false;
  if (group == 64) return !any_m_route(bits, m, g, k);
  if (m <= 16) return false;
  long long rows = 0;
  for (int i = 0; i < g.nseg; ++i) rows += g.n[i];
  if (k > kMmMaxK) return m >= 24;
  return m > 32 || rows > (kpad(k) == 3072 ? kTileRows3 : kTileRows);
}

bool group_ok(int k, int group) { return (group == 64 || group == 128) && k % group == 0 && k % 32 == 0; }

Segs make_segs(int nseg, const void* const* wt, const void* const* st, void* const* y, const int* n, const int* ldy,
               int pad) {
  Segs g;
  memset(&g, 0, sizeof(g));
  g.nseg = nseg;
  for (int i = 0, e = 0; i < nseg; ++i) {
    g.wt[i] = wt[i];
    g.st[i] = static_cast<const uint16_t*>(st[i]);
    g.y[i] = static_cast<uint16_t*>(y[i]);
    g.n[i] = n[i];
    g.ldy[i] = ldy ? ldy[i] : n[i];
    e += (n[i] + pad - 1) / pad * pad;
    g.end[i] = e;
  }
  return g;
}

// Two tokens on the wide linears go to the tokens-in-A-rows kernel (one MFMA row group holds both tokens) instead of
// the line-load kernel (one token pass per token): measured at 2 tokens, gate_up W2 55296 x 5120 25.0 -> 18.6 us, the
// LM head W4 152064 x 5120 71.5 -> 67.2 us; gate_up W3 / W4 even (27.4 / 27.7 against 27.7 / 28.4), and the
// narrow QKV, O and down slower there (10.5 -> 13.0, 8.8 -> 12.0, 18.3 -> 22.1 us).  The same bits either way.
bool two_tokens_on_mt(int bits, int m, const Segs& g) {
  if (m != 2) return false;
  long long rows = 0;
  for (int i = 0; i < g.nseg; ++i) rows += g.n[i];
  return rows >= 100000 || (bits == 2 && rows >= 32768);
}

// the default path for m <= 16 tokens: 9..16 tokens in one launch of the tokens-in-A-rows kernel where it takes them,
// else in launches of at most 8: one or two tokens on the line-load kernel
// (wq_i8m1d.hip) when their activations fit the LDS (measured faster there), otherwise and for 3..8 tokens the
// tokens-in-A-rows kernel (wq_i8mt.hip; activations beyond the LDS in chunks of stripes), and the any-m kernel
// (wq_i8.hip) for what neither takes (group 64).  act = 1 (x = gate_up [m][2k], activations SiLU(gate) * up): the
// any-m kernel does not take it (AK_INVALID).
int run_i8(int bits, const void* x, int m, const Segs& g, int k, int group, hipStream_t s, int act = 0) {
  if (m > 8) {  // 9..16 tokens in one launch of the tokens-in-A-rows kernel when it takes them
    const int e = i8_gemv_mt(bits, x, m, g, k, group, s, act);
    if (e != AK_INVALID) return e;
  }
  const size_t xk = act ? 2 * (size_t)k : (size_t)k;  // x's token stride
  const int mt = m <= 8 ? m : (m + 1) / 2;
  bool ok = true;
  for (int m0 = 0; m0 < m && ok; m0 += mt) {
    const int mm = m - m0 < mt ? m - m0 : mt;
    Segs gg = g;
    for (int i = 0; i < g.nseg; ++i) gg.y[i] = g.y[i] + (size_t)m0 * g.ldy[i];
    const void* xx = static_cast<const uint16_t*>(x) + (size_t)m0 * xk;
    int e = mm <= 2 && !two_tokens_on_mt(bits, mm, g) ? i8_gemv_m1(bits, xx, mm, gg, k, group, s, act) : AK_INVALID;
    if (e == AK_INVALID) e = i8_gemv_mt(bits, xx, mm, gg, k, group, s, act);
    if (e == AK_INVALID) e = i8_gemv_m1(bits, xx, mm, gg, k, group, s, act);
    if (e == AK_INVALID && m0 == 0) {
      ok = false;
    } else if (e) {
      return e;
    }
  }
  if (ok) return 0;
  if (act) return AK_INVALID;
  return i8_gemv(bits, x, m, g, k, group, s);
}

int gemv(int bits, const void* x, int m, int nseg, const void* const* wt, const void* const* st, void* const* y,
         const int* n, const int* ldy, int k, int group, int bf16w, bool force_default, hipStream_t s, int act = 0) {
  if (!group_ok(k, group) || nseg < 1 || nseg > kMaxSegs || m < 1 || m > 128) return AK_INVALID;
  if (bits < 2 || bits > 4 || !x || !wt || !st || !y || !n) return AK_INVALID;
  for (int i = 0; i < nseg; ++i)
    if (n[i] < 1 || !wt[i] || !st[i] || !y[i] || (ldy && ldy[i] < n[i])) return AK_INVALID;
  const bool exact = bf16w || (!force_default && exact_mode());
  if (act && exact) return AK_INVALID;  // the fused activation is in the default path's kernels only
  std::lock_guard<std::mutex> lock(scratch_mutex(s));
  const Segs all = make_segs(nseg, wt, st, y, n, ldy, 16);
  if (tile_route(bits, m, all, k, group, exact)) {
    const int e = tile_gemv(bits, x, m, all, k, group, s, act);
    if (e != AK_INVALID) return e;
  }
  if (mm_route(m, k, group, exact)) {  // above the crossover: the fp16-MFMA kernel, all tokens at once
    const int e = mm_gemv(bits, x, m, all, k, group, s, act);
    if (e != AK_INVALID) return e;
  }
  for (int m0 = 0; m0 < m; m0 += kMaxTokensPerLaunch) {
    const int mm = m - m0 < kMaxTokensPerLaunch ? m - m0 : kMaxTokensPerLaunch;
    void* yy[kMaxSegs];
    for (int i = 0; i < nseg; ++i)
      yy[i] = static_cast<uint16_t*>(y[i]) + (size_t)m0 * (ldy ? ldy[i] : n[i]);
    const void* xx = static_cast<const uint16_t*>(x) + (size_t)m0 * (act ? 2 * (size_t)k : (size_t)k);
    const int e = exact ? exact_gemv(bits, xx, mm, make_segs(nseg, wt, st, yy, n, ldy, 1), k, group, bf16w, s)
                        : run_i8(bits, xx, mm, make_segs(nseg, wt, st, yy, n, ldy, 16), k, group, s, act);
    if (e) return e;
  }
  return 0;
}

// A chain of GEMV steps: the device step table of the chained kernel, or (table == nullptr) the steps themselves, run
// one launch each.
struct Chain {
  int nsteps = 0, mt = 1;
  int kind = 0;  // 1: the one- and two-token chained kernel (wq_i8m1d.hip), 2: the 1..8-token one (wq_i8mt.hip)
  size_t smem = 0;
  void* table = nullptr;
  ak_wq_step* steps = nullptr;
};

int step_args_ok(const ak_wq_step& st) {
  if (!group_ok(st.k, st.group) || st.nseg < 1 || st.nseg > kMaxSegs || st.m < 1 || st.m > 128) return 0;
  if (st.bits < 2 || st.bits > 4 || !st.x || st.act < 0 || st.act > 1) return 0;
  for (int i = 0; i < st.nseg; ++i)
    if (st.n[i] < 1 || !st.wt[i] || !st.st[i] || !st.y[i] || (st.ldy[i] && st.ldy[i] < st.n[i])) return 0;
  return 1;
}

int run_step(const ak_wq_step& st, hipStream_t s) {
  int ldy[kMaxSegs];
  for (int i = 0; i < st.nseg; ++i) ldy[i] = st.ldy[i] ? st.ldy[i] : st.n[i];
  return gemv(st.bits, st.x, st.m, st.nseg, st.wt, st.st, st.y, st.n, ldy, st.k, st.group, st.bf16w, false, s, st.act);
}

// ---- the entry point that allocates nothing: split-K partials and counters in a static device array
//
// Bytes of split-K scratch the call's route can ask for (the tiled kernel's partials and activations are no part of it:
// where they do not fit the array, the call takes the route below it): 4 KB of row-range counters, then P (<= 8) stripe partials per
// token per output row (rows padded to 16-row blocks), 4 bytes each.  Tokens per launch: the integer kernels take at
// most 16 (padded to T = 4, 8 or 16: their token groups), the fp16-MFMA route (default numerics, group 128, m at or
// above its crossover) 16 or 32 (one or two 16-token tiles); chunks of tokens reuse the scratch in stream order.
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
__device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

size_t noalloc_scratch_need(int m, int nseg, const int* n, int k, int group, int bf16w) {
  const int tiles = kpad(k) / 1024, P = tiles < 8 ? tiles : 8;
  const bool mm = mm_route(m, k, group, bf16w || exact_mode());
  const int mt = m < 16 ? m : 16;
  const int T = mm ? (m <= 16 ? 16 : 32) : mt <= 4 ? 4 : mt <= 8 ? 8 : 16;
  size_t blocks = 0;
  for (int i = 0; i < nseg; ++i) blocks += (size_t)(n[i] + 15) / 16;
  return 4096 + (size_t)P * T * blocks * 16 * 4;
}

__global__ void zero_words_kernel(uint32_t* p, int nwords) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += gridDim.x * blockDim.x) p[i] = 0u;
}

// The device address of `scratch` on the current device (hipGetSymbolAddress once per device, with that device
// current), and at that first call its counter words cleared by a fill kernel on `s` (the kernels return every counter
// to zero at the end of each launch).  In host code `scratch` itself is only a stand-in: kernels get this address.
int noalloc_scratch(hipStream_t s, void** out) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  int dev = 0;
  int e = (int)hipGetDevice(&dev);
  if (e) return e;
  if (dev < 0 || dev >= kMaxDevices) return AK_INVALID;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    e = (int)hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e) return e;
    hipLaunchKernelGGL(zero_words_kernel, dim3(4), dim3(256), 0, s, static_cast<uint32_t*>(p), 4096 / 4);
    e = (int)hipGetLastError();
    if (e) return e;
    addr[dev] = p;
  }
  *out = addr[dev];
  return 0;
}

// One chained launch at a time per device: the chained kernel's workgroups wait on the device's flag words, which
// every chained launch on the device shares.  Launches on one stream are ordered by the stream; a launch on another
// stream is refused (hipErrorNotReady) while the device's last chained launch, issued on a different stream, has not
// finished.  Under stream capture nothing is checked or recorded (the graph's order is the caller's).
struct ChainGuard {
  static constexpr int kMaxDevices = 64;
  struct Last {
    hipStream_t stream = nullptr;
    hipEvent_t done = nullptr;
    bool recorded = false;
  };
  static std::mutex& mu() {
    static std::mutex m;
    return m;
  }
  static Last& last(int dev) {
    static Last l[kMaxDevices];
    return l[dev];
  }
  int dev = -1;
  bool capturing = false;
  std::unique_lock<std::mutex> lock;

  int begin(hipStream_t s) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (const int e = (int)hipStreamIsCapturing(s, &cs)) return e;
    capturing = cs != hipStreamCaptureStatusNone;
    if (capturing) return 0;
    if (const int e = (int)hipGetDevice(&dev)) return e;
    if (dev < 0 || dev >= kMaxDevices) return AK_INVALID;
    lock = std::unique_lock<std::mutex>(mu());
    Last& l = last(dev);
    if (l.recorded && l.stream != s) {
      const hipError_t q = hipEventQuery(l.done);
      if (q == hipErrorNotReady) return (int)hipErrorNotReady;
      if (q != hipSuccess) return (int)q;
    }
    return 0;
  }
  int end(hipStream_t s) {
    if (capturing) return 0;
    Last& l = last(dev);
    if (!l.done)
      if (const int e = (int)hipEventCreateWithFlags(&l.done, hipEventDisableTiming)) return e;
    if (const int e = (int)hipEventRecord(l.done, s)) return e;
    l.stream = s;
    l.recorded = true;
    return 0;
  }
};

}  // namespace
}  // namespace agq

using namespace agq;

extern "C" {

int ak_wq_gemv_kt_multi(int bits, const void* x, int m, int nseg, const void* const* wt, const void* const* st,
                        void* const* y, const int* n, const int* ldy, int k, int group, int bf16w, void* stream) {
  return gemv(bits, x, m, nseg, wt, st, y, n, ldy, k, group, bf16w, false, static_cast<hipStream_t>(stream));
}

// ak_wq_gemv_kt_multi that allocates nothing (no counterpart in the reference; for callers that cannot allocate: code
// under stream capture, tight serving loops): its split-K partials and the tiled kernel's converted activations lie in
// the library's static 64 MiB device array instead of library scratch.  1 (invalid value) when the call's worst-case
// split-K scratch (noalloc_scratch_need) exceeds it, e.g. a 152064-row linear at 16 tokens.  Calls on one device share
// the array: calls that overlap in time on one device race.
int ak_wq_gemv_kt_multi_noalloc(int bits, const void* x, int m, int nseg, const void* const* wt, const void* const* st,
                                void* const* y, const int* n, const int* ldy, int k, int group, int bf16w,
                                void* stream) {
  if (nseg < 1 || nseg > kMaxSegs || !n || m < 1 || k < 1) return AK_INVALID;
  for (int i = 0; i < nseg; ++i)
    if (n[i] < 1) return AK_INVALID;
  if (noalloc_scratch_need(m, nseg, n, k, group, bf16w) > kNoAllocScratchBytes) return AK_INVALID;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  void* p = nullptr;
  if (const int e = noalloc_scratch(s, &p)) return e;
  ScratchOverride& o = scratch_override();
  o = {p, kNoAllocScratchBytes, true};
  const int e = gemv(bits, x, m, nseg, wt, st, y, n, ldy, k, group, bf16w, false, s);
  o = ScratchOverride();
  return e;
}

int ak_wq_gemv_kt_silu(int bits, const void* gate_up, int m, const void* wt, const void* st, void* y, int n, int ldy,
                       int inter, int group, void* stream) {
  const int ld = ldy ? ldy : n;
  return gemv(bits, gate_up, m, 1, &wt, &st, &y, &n, &ld, inter, group, 0, false, static_cast<hipStream_t>(stream), 1);
}

int ak_w4_gemv_kt(const void* x, const void* wt, const void* st, void* y, int n, int k, int group, int bf16w,
                  void* stream) {
  return ak_wq_gemv_kt_multi(4, x, 1, 1, &wt, &st, &y, &n, nullptr, k, group, bf16w, stream);
}

int ak_w4_gemv_kt_multi(const void* x, int nseg, const void* const* wt, const void* const* st, void* const* y,
                        const int* n, int k, int group, int bf16w, void* stream) {
  return ak_wq_gemv_kt_multi(4, x, 1, nseg, wt, st, y, n, nullptr, k, group, bf16w, stream);
}

int ak_w4_gemv_kt_batched(const void* x, const void* wt, const void* st, void* y, int m, int n, int k, int group,
                          int bf16w, void* stream) {
  return ak_wq_gemv_kt_multi(4, x, m, 1, &wt, &st, &y, &n, nullptr, k, group, bf16w, stream);
}

int ak_w3_gemv_kt(const void* x, const void* wt, const void* st, void* y, int n, int k, int group, void* stream) {
  return ak_wq_gemv_kt_multi(3, x, 1, 1, &wt, &st, &y, &n, nullptr, k, group, 0, stream);
}

int ak_w3_gemv_kt_multi(const void* x, int nseg, const void* const* wt, const void* const* st, void* const* y,
                        const int* n, int k, int group, void* stream) {
  return ak_wq_gemv_kt_multi(3, x, 1, nseg, wt, st, y, n, nullptr, k, group, 0, stream);
}

int ak_w3_gemv_kt_batched(const void* x, const void* wt, const void* st, void* y, int m, int n, int k, int group,
                          void* stream) {
  return ak_wq_gemv_kt_multi(3, x, m, 1, &wt, &st, &y, &n, nullptr, k, group, 0, stream);
}

// always the default (integer MFMA) numerics, whatever ak_w4_set_mma selected
int ak_w4_mma_gemv(const void* x, const void* wt, const void* st, void* y, int m, int n, int k, int group,
                   void* stream) {
  return gemv(4, x, m, 1, &wt, &st, &y, &n, nullptr, k, group, 0, true, static_cast<hipStream_t>(stream));
}

// g128 KT conveniences of the reference: the exact numerics (their bits are the reference's tuning variants' bits)
int ak_w4g128_gemv_kt_variant(int variant, const void* x, const void* wt, const void* st, void* y, int n, int k,
                              void* stream) {
  if (k % 128 != 0) return AK_INVALID;
  switch (variant) {
    case 11: case 12: case 21: case 22: case 41: break;
    default: return AK_INVALID;
  }
  const Segs g = make_segs(1, &wt, &st, &y, &n, nullptr, 1);
  return exact_gemv(4, x, 1, g, k, 128, 0, static_cast<hipStream_t>(stream));
}

int ak_w4g128_gemv_kt_bf16(const void* x, const void* wt, const void* st, void* y, int n, int k, void* stream) {
  return ak_w4g128_gemv_kt_variant(21, x, wt, st, y, n, k, stream);
}

int ak_w4g128_gemv_kt_tune(int r, int u, int warps, int bps, const void* x, const void* wt, const void* st, void* y,
                           int n, int k, void* stream) {
  if ((r != 1 && r != 2 && r != 4) || (u != 1 && u != 2 && u != 4) || (warps != 4 && warps != 8 && warps != 16) ||
      bps < 0)
    return AK_INVALID;
  return ak_w4g128_gemv_kt_variant(11, x, wt, st, y, n, k, stream);
}

int ak_w4g128_gemv_bf16_variant(int variant, const void* x, const int32_t* packed, const void* scales, void* y, int n,
                                int k, void* stream) {
  if (k % 128 != 0 || n < 1) return AK_INVALID;
  switch (variant) {
    case 11: case 12: case 14: case 21: case 22: case 41: case 42: break;
    default: return AK_INVALID;
  }
  return exact_ct_gemv(x, packed, scales, y, n, k, static_cast<hipStream_t>(stream));
}

int ak_w4g128_gemv_bf16(const void* x, const int32_t* packed, const void* scales, void* y, int n, int k,
                        void* stream) {
  return ak_w4g128_gemv_bf16_variant(22, x, packed, scales, y, n, k, stream);
}

int ak_wq_chain_create(const ak_wq_step* steps, int nsteps, void** chain) {
  if (!steps || nsteps < 1 || !chain) return AK_INVALID;
  for (int i = 0; i < nsteps; ++i)
    if (!step_args_ok(steps[i])) return AK_INVALID;
  Chain* c = new (std::nothrow) Chain;
  if (!c) return AK_OOM;
  c->nsteps = nsteps;
  c->steps = static_cast<ak_wq_step*>(malloc(sizeof(ak_wq_step) * (size_t)nsteps));
  if (!c->steps) {
    delete c;
    return AK_OOM;
  }
  memcpy(c->steps, steps, sizeof(ak_wq_step) * (size_t)nsteps);
  // the chained kernels take default-numerics steps of group 128 (the same bits as one launch per step): at most two
  // tokens the one-token kernel's steps, up to 4 tokens (no SiLU(gate) * up step) the tokens-in-A-rows kernel's; any
  // other chain runs one launch per step
  bool chainable = !exact_mode(), small = true, act_any = false;
  for (int i = 0; i < nsteps && chainable; ++i) {
    chainable = steps[i].bf16w == 0 && steps[i].group == 128 && steps[i].m <= 4;
    small = small && steps[i].m <= 2;
    act_any = act_any || steps[i].act;
  }
  if (chainable && !small && act_any) chainable = false;
  if (chainable) {
    int* ib = static_cast<int*>(malloc(sizeof(int) * 5 * (size_t)nsteps));
    const void** xs = static_cast<const void**>(malloc(sizeof(void*) * (size_t)nsteps));
    Segs* sg = static_cast<Segs*>(malloc(sizeof(Segs) * (size_t)nsteps));
    int e = ib && xs && sg ? 0 : AK_OOM;
    if (!e) {
      int *bits = ib, *m = ib + nsteps, *k = ib + 2 * nsteps, *wait = ib + 3 * nsteps, *act = ib + 4 * nsteps;
      for (int i = 0; i < nsteps; ++i) {
        const ak_wq_step& st = steps[i];
        int ldy[kMaxSegs];
        for (int j = 0; j < st.nseg; ++j) ldy[j] = st.ldy[j] ? st.ldy[j] : st.n[j];
        bits[i] = st.bits, m[i] = st.m, k[i] = st.k, wait[i] = !st.independent, xs[i] = st.x, act[i] = st.act;
        sg[i] = make_segs(st.nseg, st.wt, st.st, st.y, st.n, ldy, 16);
      }
      e = small ? m1d_chain_make(nsteps, bits, xs, m, k, sg, wait, act, &c->table, &c->mt, &c->smem)
                : mt_chain_make(nsteps, bits, xs, m, k, sg, wait, &c->table, &c->mt, &c->smem);
      c->kind = e ? 0 : small ? 1 : 2;
    }
    free(ib);
    free(xs);
    free(sg);
    if (e && e != AK_INVALID) {  // AK_INVALID: a step does not suit the chained kernel (one launch per step)
      free(c->steps);
      delete c;
      return e;
    }
  }
  *chain = c;
  return 0;
}

int ak_wq_chain_run(void* chain, void* stream) {
  if (!chain) return AK_INVALID;
  const Chain* c = static_cast<const Chain*>(chain);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (c->table) {
    ChainGuard g;
    if (const int e = g.begin(s)) return e;
    const int e = c->kind == 1 ? m1d_chain_launch(c->table, c->nsteps, c->mt, c->smem, s)
                               : mt_chain_launch(c->table, c->nsteps, c->mt, c->smem, s);
    return e ? e : g.end(s);
  }
  for (int i = 0; i < c->nsteps; ++i)
    if (const int e = run_step(c->steps[i], s)) return e;
  return 0;
}

int ak_wq_chain_chained(void* chain) { return chain && static_cast<const Chain*>(chain)->table ? 1 : 0; }

int ak_wq_chain_destroy(void* chain) {
  if (!chain) return 0;
  Chain* c = static_cast<Chain*>(chain);
  const int e = c->table ? (int)hipFree(c->table) : 0;
  free(c->steps);
  delete c;
  return e;
}

int ak_wq_chain_status(void) {
  int err = 0, err2 = 0;
  int e = m1d_chain_error(&err);
  if (!e) e = mt_chain_error(&err2);
  return e ? -e : (err || err2 ? 1 : 0);
}

int ak_wq_tune_override(int split, int nwv, int sk) {
  m1d_tune_override(split, nwv, sk < -2 ? -1 : sk > 1 ? 1 : sk);
  return 0;
}

int ak_wq_tune_query(int bits, int m, int nseg, const int* n, int k, int* split, int* nwv, int* sk) {
  if (!n || !split || !nwv || !sk || nseg < 1 || nseg > kMaxSegs || !group_ok(k, 128)) return AK_INVALID;
  for (int i = 0; i < nseg; ++i)
    if (n[i] < 1) return AK_INVALID;
  void* dummy[kMaxSegs] = {};
  const Segs g = make_segs(nseg, dummy, dummy, dummy, n, nullptr, 16);
  return m1d_tune_query(bits, m, g, k, split, nwv, sk);
}

int ak_wq_set_mm_min(int m) {
  g_mm_min.store(m < 0 ? -1 : m, std::memory_order_relaxed);
  return 0;
}

int ak_w4_set_mma(int mode) {
  g_mode.store(mode < 0 ? -1 : (mode ? 1 : 0), std::memory_order_relaxed);
  return 0;
}
// reference: selects a bit-identical sm90 kernel variant; one default kernel family here, so accepted and ignored
int ak_w4_set_lean(int rb) {
  (void)rb;
  return 0;
}
int ak_w4_set_tma(int stages) {
  (void)stages;
  return 0;
}

}  // extern "C"
