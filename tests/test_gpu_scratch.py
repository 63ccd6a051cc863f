"""Calls that work in library scratch (the tiled GEMV and the k-split prefill GEMM) at once on streams whose kernels
nothing orders: every call's outputs are the ones it gives alone, bit for bit."""
import ctypes
import threading

import numpy as np
import pytest

from _lib import kernels, check, Dev, Linear, gen_container, gen_scales, gen_x, ptr_array, int_array

pytestmark = pytest.mark.gpu

vp = ctypes.c_void_p
PER_THREAD = vp(2)  # hipStreamPerThread


@pytest.fixture(scope="module")
def gpu():
    K = kernels()
    n = ctypes.c_int(0)
    assert K.ak_device_count(ctypes.byref(n)) == 0 and n.value >= 1, "no GPU visible"
    K.ak_w4_set_mma(1)
    yield K, ctypes.CDLL("libamdhip64.so")
    K.ak_w4_set_mma(-1)


class Call:
    """One GEMV (or, `gemm`, one prefill GEMM) on inputs of its own and its outputs when nothing else runs."""

    def __init__(self, K, seed, group, bits, m, n, k, gemm=False):
        self.K, self.L, self.gemm = K, Linear(gen_container(seed, n, k, -(1 << (bits - 1)), 1 << bits),
                                              gen_scales(seed + 1, n * k // group), n, k, group, bits), gemm
        check(self.L.rc, "repack")
        self.m, self.X, self.Y = m, Dev.of(gen_x(seed + 2, m * k)), Dev(m * n * 2)
        self.rc = self.enqueue(None)
        check(self.rc)
        self.want = self.out()

    def enqueue(self, stream):
        L = self.L
        if self.gemm:
            return self.K.ak_wq_gemm_kt(L.bits, self.X.p, self.m, L.wt.p, L.st.p, self.Y.p, L.n, 0, L.k, L.group, stream)
        return self.K.ak_wq_gemv_kt_multi(L.bits, self.X.p, self.m, 1, ptr_array([L.wt.p]), ptr_array([L.st.p]),
                                          ptr_array([self.Y.p]), int_array([L.n]), None, L.k, L.group, 0, stream)

    def clear(self):
        junk = np.full(self.m * self.L.n, 0x7FC1, dtype=np.uint16)
        check(self.K.ak_memcpy_h2d(self.Y.p, junk.ctypes.data, junk.nbytes), "h2d")

    def out(self):
        check(self.K.ak_synchronize(), "sync")
        return self.Y.get(np.uint16, self.m * self.L.n)


# (group, bits, tokens, rows, inputs): unsplit (the activations alone in scratch), split (partials and counters too)
SHAPES = [(64, 4, 3, 20000, 1024), (64, 4, 2, 600, 6144), (128, 3, 40, 14000, 1024), (128, 2, 64, 600, 9344)]


@pytest.mark.parametrize("group,bits,m,n,k", SHAPES)
def test_two_threads_on_the_per_thread_stream(gpu, group, bits, m, n, k):
    K, hip = gpu
    calls = [Call(K, 100 + 10 * i, group, bits, m, n, k) for i in range(2)]
    for c in calls:
        c.clear()
    rcs, meet = [], threading.Barrier(2)

    def work(c):
        rcs.append(c.enqueue(PER_THREAD))  # the first call allocates and synchronizes
        rcs.append(hip.hipStreamSynchronize(PER_THREAD))
        meet.wait()
        for _ in range(40):
            rcs.append(c.enqueue(PER_THREAD))
        rcs.append(hip.hipStreamSynchronize(PER_THREAD))

    threads = [threading.Thread(target=work, args=(c,)) for c in calls]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not any(rcs)
    for c in calls:
        assert np.array_equal(c.out(), c.want)


def capture(hip, stream, enqueue):
    graph, exe = vp(), vp()
    assert hip.hipStreamBeginCapture(stream, ctypes.c_int(1)) == 0
    rc = enqueue(stream)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    check(rc, "under capture")
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    return graph, exe


def nodes(hip, graph):
    n = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("group,bits,m,n,k,gemm", [s + (False,) for s in SHAPES] + [(128, 2, 200, 640, 9344, True)])
def test_two_graphs_and_a_call_at_once(gpu, group, bits, m, n, k, gemm, warm):
    """Two graphs captured from one stream (that the library has worked on before, or not), replayed on two others while
    the stream itself runs a third call: several replays, each as the call alone."""
    K, hip = gpu
    calls = [Call(K, 300 + 10 * i, group, bits, m, n, k, gemm) for i in range(3)]
    streams = [vp() for _ in range(3)]
    for s in streams:
        assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    if warm:
        check(calls[2].enqueue(streams[2]))
        assert hip.hipStreamSynchronize(streams[2]) == 0
    graphs = [capture(hip, streams[2], c.enqueue) for c in calls[:2]]
    assert all(nodes(hip, g) == 2 for g, _ in graphs), "the two kernels of the route that needs scratch"
    check(calls[2].enqueue(streams[2]))  # (its first call allocates and synchronizes)
    for rep in range(4):
        for c in calls:
            c.clear()
        check(K.ak_synchronize())
        for _ in range(8):
            for (_, e), s in zip(graphs, streams):
                assert hip.hipGraphLaunch(e, s) == 0
            check(calls[2].enqueue(streams[2]))
        for i, c in enumerate(calls):
            assert np.array_equal(c.out(), c.want), f"replay {rep}, call {i}"
    for g, e in graphs:
        hip.hipGraphExecDestroy(e)
        hip.hipGraphDestroy(g)
    for s in streams:
        hip.hipStreamDestroy(s)
