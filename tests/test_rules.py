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
