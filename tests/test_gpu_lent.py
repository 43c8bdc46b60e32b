"""Device buffers that tg_buffer lends, with the caller's own work on them (through the HIP
runtime that libtagore.so links; no torch in this process)."""
import ctypes

import numpy as np
import pytest

import oracle
import tagore_amd
from tagore_amd import State
from tests.conftest import gmm_int, gmm_unit

pytestmark = pytest.mark.gpu

H2D = 1  # hipMemcpyHostToDevice


def _hip():
    tagore_amd.lib()  # loads libamdhip64.so.7 as libtagore.so's dependency
    h = ctypes.CDLL("libamdhip64.so.7")
    h.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    return h


@pytest.mark.parametrize("first,second", [("u8", "u8"), ("u8", "real"), ("real", "real")])
def test_vectors_written_through_the_lent_buffer(first, second):
    """Vectors replaced through the device pointer after calls that prepared the first ones: the
    search, the prune and the build that follow use the new vectors."""
    hip = _hip()
    N, D, K, FD = 1200, 64, 24, 16
    make = {"u8": lambda seed: gmm_int(N, D, 8, seed), "real": lambda seed: gmm_unit(N, D, 8, seed)}
    X1, X2 = make[first](1), make[second](2)
    Q = make[first](3)[:40].copy()
    with State(N, D) as s:
        s.set_data(X1)
        s.knn_build(K, 4, 5, "bf16")
        s.prune("path", "dist", "dist", FD, 32, 1.2)
        deg, ids, ep = s.get_pruned()
        ptr, nbytes = s.buffer(2)
        assert nbytes == X2.nbytes
        assert hip.hipMemcpy(ptr, X2.ctypes.data, X2.nbytes, H2D) == 0
        print(f"lent vectors {first} -> {second}", flush=True)
        oi, od, oc = oracle.search(X2, deg, ids, ep, Q, 32, 10, 0x44)
        gi, gd, st = s.search(Q, k=10, L=32, seed=0x44)
        assert np.array_equal(gi, oi) and np.array_equal(gd, od) and st["evals"] == oc["evals"]
        G, GD = oracle.knn_bruteforce(X2, K)
        s.set_knn(G, GD)
        ref = oracle.prune(X2, G, GD, FD, 32, 0, 0, 0, 1.2)
        for rep in range(2):
            s.prune("path", "dist", "dist", FD, 32, 1.2)
            rdeg, rids, rep_ = s.get_pruned()
            assert rep_ == ref["ep"] and np.array_equal(rdeg, ref["deg"])
            for u in range(N):
                assert np.array_equal(rids[u, :rdeg[u]], ref["ids"][u, :rdeg[u]])
        Gr, GDr, _ = oracle.gnn_descent(X2, K, 4, 5)
        for prec in ("fp32", "bf16", "fp8"):
            s.knn_build(K, 4, 5, prec)
            G, GD = s.get_knn()
            assert np.array_equal(G, Gr) and np.array_equal(GD, GDr), prec
        s.set_data(X1)
        s.set_pruned(deg, ids, ep)
        oi, od, oc = oracle.search(X1, deg, ids, ep, Q, 32, 10, 0x44)
        gi, gd, st = s.search(Q, k=10, L=32, seed=0x44)
        assert np.array_equal(gi, oi) and np.array_equal(gd, od)


@pytest.mark.parametrize("own_stream", [False, True])
@pytest.mark.parametrize("N", [1000, 1 << 19])
def test_results_follow_the_callers_work_on_lent_lists(N, own_stream):
    """New distances written into the lent lists by the caller's asynchronous copies on the
    default stream, or on a stream that the default one waits for, with other work before
    them: the copy to the host (plain, and by chunks) comes after them."""
    hip = _hip()
    vp = ctypes.c_void_p
    hip.hipMalloc.argtypes = [ctypes.POINTER(vp), ctypes.c_size_t]
    hip.hipFree.argtypes = [vp]
    hip.hipMemcpyAsync.argtypes = [vp, vp, ctypes.c_size_t, ctypes.c_int, vp]
    hip.hipStreamCreate.argtypes = [ctypes.POINTER(vp)]
    hip.hipStreamDestroy.argtypes = [vp]
    hip.hipStreamSynchronize.argtypes = [vp]
    K, big, D2D = 4, 256 << 20, 3
    rng = np.random.default_rng(N)
    ids = rng.integers(0, N, (N, K)).astype(np.uint32)
    d1 = (np.arange(K) + 0.5 * rng.random((N, K))).astype(np.float32)
    d2 = (np.arange(K) + 0.5 * rng.random((N, K))).astype(np.float32)
    src, a, b, stream = vp(), vp(), vp(), vp()
    assert hip.hipMalloc(ctypes.byref(src), d2.nbytes) == 0
    assert hip.hipMalloc(ctypes.byref(a), big) == 0 and hip.hipMalloc(ctypes.byref(b), big) == 0
    if own_stream:
        assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    with State(N, 4) as s:
        s.set_knn(ids, d1)
        s.get_knn()
        ptr, nbytes = s.buffer(3)
        assert nbytes == d2.nbytes
        assert hip.hipMemcpy(src, d2.ctypes.data, d2.nbytes, H2D) == 0
        print(f"lent lists N={N} own stream {own_stream}", flush=True)
        for _ in range(100):  # some 10 ms before the lists change
            assert hip.hipMemcpyAsync(a, b, big, D2D, stream) == 0
        assert hip.hipMemcpyAsync(ptr, src, d2.nbytes, D2D, stream) == 0
        G, GD = s.get_knn()
        assert np.array_equal(G, ids) and np.array_equal(GD, d2)
        assert hip.hipStreamSynchronize(stream) == 0
    for p in (src, a, b):
        assert hip.hipFree(p) == 0
    if own_stream:
        assert hip.hipStreamDestroy(stream) == 0


def test_search_gives_large_buffers_back():
    """A search over many queries leaves no more than its bound of device memory with the
    handle (2 x 64 MiB); small and large calls in turn answer alike."""
    hip = _hip()
    hip.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t), ctypes.POINTER(ctypes.c_size_t)]

    def free_bytes():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    rng = np.random.default_rng(3)
    N, D, nq = 500, 256, 400_000  # queries of 410 MB, results of 160 MB at k = 50
    X = rng.integers(0, 256, (N, D)).astype(np.float32)
    Q = X[rng.integers(0, N, nq)]
    ids = rng.integers(0, N, (N, 4)).astype(np.uint32)
    with State(N, D) as s:
        s.set_data(X)
        s.set_pruned(np.full(N, 4, np.uint32), ids, 0)
        small = s.search(Q[:20], k=50, L=50, seed=1)
        before = free_bytes()
        for rep in range(2):
            print(f"large search {rep}", flush=True)
            large = s.search(Q, k=50, L=50, seed=1)
            assert before - free_bytes() <= 128 << 20
            assert np.array_equal(large[0][:20], small[0]) and np.array_equal(large[1][:20], small[1])
            again = s.search(Q[:20], k=50, L=50, seed=1)
            assert np.array_equal(again[0], small[0]) and np.array_equal(again[1], small[1])
