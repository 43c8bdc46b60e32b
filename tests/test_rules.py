"""Bounds and launch rules of the host side (tagore_amd/csrc/rules.hpp), compiled with the host
compiler: no GPU needed."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tests.conftest import ROOT

SRC = """
#include "rules.hpp"
extern "C" float kappa16(double rho, uint32_t D, uint32_t chain) {
  return tg::screen_kappa16(rho, D, chain);
}
extern "C" uint32_t hash_bits(uint32_t L, uint32_t FD, uint32_t per_cu) {
  return tg::search_hash_bits(L, FD, per_cu);
}
extern "C" uint32_t search_lds() { return tg::SEARCH_LDS; }
extern "C" float kappa32(uint32_t D) { return tg::screen_kappa32(D); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SRC)
    out = str(d / "rules.so")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I",
                           os.path.join(ROOT, "tagore_amd", "csrc"), str(d / "rules.cpp"), "-o", out])
    L = ctypes.CDLL(out)
    L.kappa16.restype = L.kappa32.restype = ctypes.c_float
    L.kappa16.argtypes = [ctypes.c_double, ctypes.c_uint32, ctypes.c_uint32]
    L.kappa32.argtypes = [ctypes.c_uint32]
    return L


def _cut(x):
    """x to 24 bits, cut off."""
    m, e = np.frexp(x)
    return np.ldexp(np.trunc(m * 2.0**24), e - 24)


def _product(a, b, step, how):
    """sum a b as a chain of steps of `step` elements with FP32 sums."""
    acc = 0.0
    for k in range(0, len(a), step):
        p = a[k:k + step].astype(np.float64) * b[k:k + step].astype(np.float64)
        if how == "aligned":  # every addend cut to the unit of the largest
            unit = 2.0 ** (np.frexp(max(abs(acc), np.abs(p).max()))[1] - 24)
            acc = float(_cut(np.trunc(acc / unit) * unit + (np.trunc(p / unit) * unit).sum()))
        else:
            for q in p:
                acc = float(np.float32(acc + q)) if how == "nearest" else float(_cut(acc + q))
    return acc


@pytest.mark.parametrize("D", [4, 32, 96, 512, 960, 1024])
@pytest.mark.parametrize("step,chain", [(32, 1024), (32, 128), (4, 1024)])
@pytest.mark.parametrize("how", ["nearest", "cut", "aligned"])
def test_screen_slack_covers_any_accumulation(rules, D, step, chain, how):
    """One product of 1 and D - 1 just below the size that a sum of 1 keeps: the rows whose
    screen distance an FP32 accumulation can put off most.  The slack covers every order and
    rounding (values that BF16 and FP16 hold exactly), of the whole row and of chains summed."""
    small = 2.0**-12 if how == "nearest" else 2.0**-11
    a = np.full(D, small * (1 - 2.0**-8), np.float32)
    b = np.full(D, 2.0**-12, np.float32)
    for at in {0, D // 2, D - 1}:
        x, y = a.copy(), b.copy()
        x[at] = y[at] = 1.0
        na, nb = (x.astype(np.float64)**2).sum(), (y.astype(np.float64)**2).sum()
        d = ((x.astype(np.float64) - y)**2).sum()
        dot = np.float32(0)
        for k in range(0, D, chain):
            dot += np.float32(_product(x[k:k + chain], y[k:k + chain], step, how))
        s = (na + nb) - 2.0 * float(dot)
        kap = rules.kappa16(0.0, D, chain) if step == 32 else rules.kappa32(D)
        assert abs(s - d) <= kap * (na + nb), (at, abs(s - d) / (na + nb) * 2**23, kap * 2**23)


@pytest.mark.parametrize("L", [1, 10, 64, 65, 128, 256])
@pytest.mark.parametrize("FD", [1, 16, 32, 48, 96, 128])
def test_search_hash_leaves_room_for_the_workgroups(rules, L, FD):
    """A CU's 160 KB hold as many workgroups as are to run there, up to 21 (the smallest hash);
    up to four, the hash has the size that the number of visited ids asks for; the initial ids
    always fit."""
    usual = L * FD // 2 + L + 128
    want = next((b for b in range(10, 13) if 2 << b >= 3 * usual), 13)
    for per_cu in range(1, 22):
        bits = rules.hash_bits(L, FD, per_cu)
        lds = -(-((4 << bits) + rules.search_lds()) // 1280) * 1280
        assert per_cu * lds <= 160 * 1024, (per_cu, bits)
        assert bits == want if per_cu <= 4 else 10 <= bits <= want
        assert (3 << bits) // 4 >= 256 + 128
