/* libagens_kernels: tuning entry points of the one- and two-token GEMV (the role of the reference's tuning entries,
 * kernels/include/agens_kernels.h:271-277 ak_w4g128_gemv_kt_tune / _variant and the launch pins of
 * tools/aot_pins_sm90.json, produced by kernels/bench/tune_w4.cu:1-91).  Every launch configuration gives the same
 * output bits; these only select among them.  Used by agens-engine_amd/tune_launch.py, which measures the candidates
 * and writes the compiled-in table (csrc/wq_launch_table.h) that ak_wq_gemv_kt_multi consults.  Not for engines:
 * every switch here is process-global (it changes the launches of every thread until it is reset) and meant for
 * tuning and tests. */
#pragma once

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Forces the launch configuration of the following one- and two-token GEMV launches (group 128, default numerics) in
 * this process: split = stripe sets per 4-row block (1, 2, 4, 8; 0: not forced), nwv = waves per workgroup (16, 8;
 * 0: not forced), sk = split-K across workgroups (1 yes, 0 no, -1 not forced, -2 not forced and the measured pins
 * ignored: the cost model alone).  A forced value the shape does not admit is ignored for that launch.  Always 0. */
int ak_wq_tune_override(int split, int nwv, int sk);

/* The configuration a one- or two-token launch (m = 1, 2) of these segments takes now (pins, override and cost model
 * applied): 0 and *split, *nwv, *sk (1: split-K across workgroups), or 1 if the shape is not one this kernel takes. */
int ak_wq_tune_query(int bits, int m, int nseg, const int* n, int k, int* split, int* nwv, int* sk);

/* The tiling of an ak_wq_gemm_kt call: rows and tokens per tile, k splits (1: none) and the bytes of scratch that the
 * splits' partial sums take.  0, or 1 for a shape that the call refuses. */
int ak_wq_gemm_tune_query(int m, int n, int k, int* rows, int* tokens, int* splits, size_t* scratch);

/* An explicit crossover between the older kernels of the default numerics, for every ak_wq_gemv_kt_multi call: at group
 * 128, m >= this many tokens take the fp16-MFMA kernel and fewer the integer-limb kernels, at every k; 0: the
 * integer-limb kernels for every m.  While one is set (a value of 0 or more, or the environment variable
 * AGENS_WQ_MM_MIN), the tiled kernel (csrc/wq_tile.h) is off at every group and token count -- also with the value 17,
 * and also at group 64, where the any-m kernel is left: up to ten times slower (16 tokens, 5120 x 6144: 188 against 19
 * us).  Negative: the compiled-in measured rules (tile_route, any_m_route and mm_route of csrc/wq_api.hip).  All of these
 * kernels compute the same numerics bit for bit, so this changes speed only.  Process-wide.  Always 0. */
int ak_wq_set_mm_min(int m);

#ifdef __cplusplus
}
#endif
