// The host library's choice of the prefill route (host/agens_linear.cpp, linear() above 128 tokens) on the CPU: the C ABI
// below records the calls.  Prints one line per failed check; exit status 0 when there is none.
#include <stdio.h>
#include <stdlib.h>

#include "agens_linear.h"

namespace {
int gemms = 0, rows = 0, products = 0, failed = 0;
constexpr long long kLimit = 1ll << 31;  // what the fused GEMM takes of weights and of activations

long long weight_bytes(int bits, int n, int k) { return (long long)((k + 1023) / 1024) * n * 128 * bits; }
void expect(bool ok, const char* what) {
  if (ok) return;
  printf("FAILED: %s\n", what);
  ++failed;
}
}  // namespace

extern "C" {
const char* ak_error_string(int) { return ""; }
int ak_malloc(void** p, size_t n) { return (*p = malloc(n)) ? 0 : 2; }
int ak_free(void* p) { return free(p), 0; }
int ak_memcpy_h2d(void*, const void*, size_t) { return 0; }
int ak_synchronize(void) { return 0; }
size_t ak_wq_kt_weight_bytes(int bits, int n, int k) { return (size_t)weight_bytes(bits, n, k); }
size_t ak_w4_kt_scale_bytes(int, int, int) { return 1; }
int ak_wq_repack_kt(int, const int32_t*, const void*, void*, void*, int, int, int, void*) { return 0; }
int ak_wq_gemm_kt(int bits, const void*, int m, const void*, const void*, void*, int n, int, int k, int, void*) {
  if (weight_bytes(bits, n, k) >= kLimit || (long long)m * k * 2 >= kLimit) return 1;
  return ++gemms, 0;
}
int ak_wq_dequant_kt_rows(int, const void*, const void*, void*, int n, int, int, int r0, int nr, void*) {
  return r0 + nr > n ? 1 : (rows += nr, 0);
}
int ak_bf16_linear_f32reduce(const void*, const void*, void*, int, int, int, void*) { return ++products, 0; }
int ak_bf16_linear_f32reduce_ld(const void*, const void*, void*, int, int, int, int, void*) { return ++products, 0; }
int ak_wq_gemv_kt_multi(int, const void*, int, int, const void* const*, const void* const*, void* const*, const int*,
                        const int*, int, int, int, void*) {
  return 0;
}
int ak_wq_chain_create(const ak_wq_step*, int, void**) { return 0; }
int ak_wq_chain_run(void*, void*) { return 0; }
int ak_wq_chain_chained(void*) { return 0; }
int ak_wq_chain_destroy(void*) { return 0; }
}

namespace {
// one part of `bits` bits: whether linear() succeeds, and by which route
void linear(int bits, int m, int n, int k, bool fused, const char* what) {
  agens::QuantLinear t;
  t.n = n, t.k = k, t.np = 1;
  t.p[0].bits = bits, t.p[0].group = 128, t.p[0].r0 = 0, t.p[0].n = n;
  static char byte;
  t.p[0].wt = t.p[0].st = &byte;
  gemms = rows = products = 0;
  expect(agens::linear(t, &byte, &byte, m, n, k, 0, nullptr) == 0, what);
  expect(fused ? gemms == 1 && !products : gemms == 0 && rows == n && products > 0, what);
}
}  // namespace

int main() {
  agens::set_prefill_tile_bytes((size_t)1 << 20);  // (the route, not the memory)
  linear(4, 512, 5120, 5120, true, "fused up to 768 tokens");
  linear(4, 769, 5120, 5120, false, "the library GEMM above");
  linear(2, 1536, 5120, 27648, true, "fused up to 1536 tokens at long k");
  linear(4, 577, 8192, 4096, false, "the library GEMM on middling rows of short k");
  linear(4, 576, 8192, 4096, true, "fused up to 576 tokens there");
  linear(4, 768, 8192, 2048, true, "and at shorter k");
  linear(4, 768, 8193, 4096, true, "and on more rows");
  // weights of 2 GB and just below, activations of 2 GB and just below, at every route's token counts
  linear(4, 1100, 131072, 32768, false, "weights of 2 GB, long k");
  linear(4, 1100, 131071, 32768, true, "weights just below");
  linear(4, 600, 262144, 16384, false, "weights of 2 GB, 600 tokens");
  linear(4, 1000, 524288, 8192, false, "weights of 2 GB, wide");
  linear(3, 1100, 131072, 32768, true, "three quarters of that");
  linear(2, 1536, 128, 699136, false, "activations of 2 GB");
  linear(2, 1535, 128, 699136, true, "activations just below");
  if (!failed) printf("route: all checks passed\n");
  return failed ? 1 : 0;
}
