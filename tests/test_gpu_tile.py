"""The tiled batched GEMV (csrc/wq_tile.h): the default numerics at more than 16 tokens and at group 64, bit for bit
against the oracle (which restates them: exact integer group sums rounded once, a fixed fp32 order), at the edges of
its token tiles, row blocks, segments, stripes and launch shapes, and against the kernels a call falls back to."""
import ctypes

import numpy as np
import pytest

from _lib import (kernels, check, Dev, Linear, gemv, gen_container, gen_scales, gen_x, ora_fast, ptr_array, int_array,
                  f2bf_array)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    K = kernels()
    n = ctypes.c_int(0)
    assert K.ak_device_count(ctypes.byref(n)) == 0 and n.value >= 1, "no GPU visible"
    K.ak_w4_set_mma(1)
    yield K
    K.ak_w4_set_mma(-1)


def make(seed, n, k, group, bits):
    L = Linear(gen_container(seed, n, k, -(1 << (bits - 1)), 1 << bits), gen_scales(seed + 1, n * k // group), n, k,
               group, bits)
    check(L.rc, "repack")
    return L


def assert_equals_oracle(y, x, m, L, spans):
    wt, st = L.host_kt()
    for r0, r1 in spans:
        want = ora_fast(L.bits, x, m, wt, st, L.n, L.k, L.group, rows=(r0, r1))[:, r0:r1]
        got = y[:, r0:r1]
        assert np.array_equal(got, want), \
            f"rows {r0}..{r1}: {int(np.sum(got != want))} differ, e.g. {np.argwhere(got != want)[:4].tolist()}"


# group, bits, tokens, segments' rows, inputs: one of each kind of edge
EDGES = [
    (128, 4, 33, (16,), 128), (128, 3, 64, (17, 1), 1024), (128, 2, 65, (1, 16, 33, 250), 1152),
    (128, 3, 128, (225,), 2048), (128, 2, 48, (80, 300), 9344), (128, 4, 127, (300,), 8320),
    (128, 3, 17, (6200,), 256), (128, 2, 32, (3000, 3150, 15), 1280), (128, 2, 24, (40,), 8320),
    (64, 4, 1, (1,), 64), (64, 4, 2, (15,), 192), (64, 3, 16, (129, 2), 1088), (64, 2, 17, (260,), 4160),
    (64, 4, 33, (113,), 1024), (64, 3, 128, (450,), 2112), (64, 2, 9, (70,), 9280),
]


@pytest.mark.parametrize("group,bits,m,ns,k", EDGES)
def test_equals_oracle_bit_for_bit(group, bits, m, ns, k):
    lins = [make(40 + 2 * i, n, k, group, bits) for i, n in enumerate(ns)]
    ldy = [n + (3 if i % 2 else 0) for i, n in enumerate(ns)]
    x = gen_x(7 + m, m * k)
    ys = gemv(bits, Dev.of(x), m, lins, k, group, ldy=ldy)
    for i, L in enumerate(lins):
        y = ys[i].get(np.uint16, m * ldy[i]).reshape(m, ldy[i])
        assert_equals_oracle(y, x, m, L, [(0, L.n)])


# wide linears: every number of row blocks per wave, more than one round of workgroups, a ragged last one
@pytest.mark.parametrize("group,bits,m,n", [(64, 4, 1, 60001), (64, 3, 20, 60001), (128, 3, 18, 60001),
                                            (128, 4, 33, 14001), (128, 2, 49, 57000), (128, 3, 64, 40001),
                                            (128, 4, 128, 28001), (128, 2, 65, 19999), (64, 2, 64, 33000)])
def test_wide_linears_equal_oracle(group, bits, m, n):
    k = 1152
    L = make(11, n, k, group, bits)
    x = gen_x(13 + m, m * k)
    (Y,) = gemv(bits, Dev.of(x), m, [L], k, group)
    y = Y.get(np.uint16, m * n).reshape(m, n)
    assert_equals_oracle(y, x, m, L, [(0, 130), (n // 2, n // 2 + 130), (n - 130, n)])


# both sides of the lines between the tiled kernel and the integer kernels (by full rounds of the latter's workgroups of
# 64 rows at group 64; above 8192 inputs at group 128)
@pytest.mark.parametrize("group,bits,m,n,k", [(64, 4, 1, 13040, 5120), (64, 4, 1, 13057, 5120), (64, 3, 1, 16384, 5184),
                                            (64, 2, 1, 32768, 5120), (64, 2, 1, 32769, 5120), (64, 3, 2, 24560, 6144),
                                            (64, 3, 2, 24576, 6144), (64, 2, 1, 16400, 8256), (64, 4, 1, 65600, 6208),
                                            (128, 2, 33, 16001, 10368), (128, 3, 41, 16001, 10368),
                                            (128, 3, 33, 10240, 10368), (128, 3, 33, 10241, 10368), (128, 4, 40, 10241, 16384),
                                            (128, 4, 41, 10241, 16384), (128, 4, 33, 10241, 16512), (128, 2, 33, 10241, 16512),
                                            (128, 2, 33, 17001, 10368), (128, 2, 41, 17001, 10368), (128, 3, 64, 12635, 6912),
                                            (128, 2, 65, 22288, 6528), (128, 3, 17, 8192, 2176), (128, 3, 32, 8193, 3072)])
def test_routes_equal_oracle(group, bits, m, n, k):
    L = make(17, n, k, group, bits)
    x = gen_x(19 + m, m * k)
    (Y,) = gemv(bits, Dev.of(x), m, [L], k, group)
    y = Y.get(np.uint16, m * n).reshape(m, n)
    assert_equals_oracle(y, x, m, L, [(0, 40), (n // 2, n // 2 + 40), (n - 40, n)])


@pytest.mark.parametrize("group,bits,m,n,k", [(128, 3, 40, 7000, 1024), (128, 2, 100, 600, 9344), (64, 4, 3, 600, 2112),
                                              (128, 2, 128, 40, 163840)])
def test_equals_the_other_kernels(group, bits, m, n, k):
    """The kernels an explicit crossover selects, the entry point without allocation (the last case's converted
    activations are larger than its array: the older kernels), and captures of a stream that the library has not worked
    on and has: the same bits; the captured launches, which are the tiled kernel's two, replay."""
    K = kernels()
    hip = ctypes.CDLL("libamdhip64.so")
    vp = ctypes.c_void_p
    L = make(21, n, k, group, bits)
    X = Dev.of(gen_x(5, m * k))

    def out(fn):
        Y = Dev.of(np.full(m * n, 0x7FC1, dtype=np.uint16))
        fn(Y)
        check(K.ak_synchronize(), "sync")
        return Y.get(np.uint16, m * n)

    def args(Y):
        return (bits, X.p, m, 1, ptr_array([L.wt.p]), ptr_array([L.st.p]), ptr_array([Y.p]), int_array([n]), None, k,
                group, 0)

    want = out(lambda Y: check(K.ak_wq_gemv_kt_multi(*args(Y), None)))
    for crossover in (0, 2):
        K.ak_wq_set_mm_min(crossover)
        try:
            assert np.array_equal(out(lambda Y: check(K.ak_wq_gemv_kt_multi(*args(Y), None))), want)
        finally:
            K.ak_wq_set_mm_min(-1)
    assert np.array_equal(out(lambda Y: check(K.ak_wq_gemv_kt_multi_noalloc(*args(Y), None))), want)
    stream = vp()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    for warm in (False, True):
        Y, graph, exe = Dev(m * n * 2), vp(), vp()
        if warm:
            check(K.ak_wq_gemv_kt_multi(*args(Y), stream))
            assert hip.hipStreamSynchronize(stream) == 0
        assert hip.hipStreamBeginCapture(stream, ctypes.c_int(1)) == 0
        rc = K.ak_wq_gemv_kt_multi(*args(Y), stream)
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        check(rc, "under capture")
        count = ctypes.c_size_t()
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0 and count.value == 2
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
        for rep in range(3):
            junk = np.full(m * n, 0x7FC1, dtype=np.uint16)
            check(K.ak_memcpy_h2d(Y.p, junk.ctypes.data, junk.nbytes), "h2d")
            assert hip.hipGraphLaunch(exe, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
            assert np.array_equal(Y.get(np.uint16, m * n), want), f"replay {rep}"
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(stream)


@pytest.mark.parametrize("bits,m,n,inter", [(2, 40, 300, 9344), (3, 65, 70, 1152), (4, 20, 7000, 256)])
def test_fused_activation_equals_silu_then_gemv(bits, m, n, inter):
    K = kernels()
    L = make(31, n, inter, 128, bits)
    X = Dev.of(f2bf_array(np.random.default_rng(m).standard_normal(2 * m * inter).astype(np.float32) * 2))
    Y, A = Dev(m * n * 2), Dev(m * inter * 2)
    check(K.ak_wq_gemv_kt_silu(bits, X.p, m, L.wt.p, L.st.p, Y.p, n, 0, inter, 128, None))
    check(K.ak_silu_mul(X.p, A.p, m, inter, None))
    (Z,) = gemv(bits, A, m, [L], inter, 128)
    check(K.ak_synchronize())
    assert np.array_equal(Y.get(np.uint16, m * n), Z.get(np.uint16, m * n))
