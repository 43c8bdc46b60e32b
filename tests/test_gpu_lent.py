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
