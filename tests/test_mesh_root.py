"""The square root of the mesh winding kernel (mpm_root.h), compiled alone: from
any estimate as far off as the device's may be, within an ulp of sqrt."""

import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent

SOURCE = r"""
#include <cstdint>
#include "mpm_root.h"
extern "C" void roots(const double* x, const double* y, double* out, uint64_t n) {
  for (uint64_t i = 0; i < n; ++i) out[i] = tmpm::refine_root(x[i], y[i]);
}
"""


@pytest.fixture(scope="module")
def roots(tmp_path_factory):
    d = tmp_path_factory.mktemp("root")
    (d / "r.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    str(ROOT / "tessera_amd" / "csrc"), str(d / "r.cpp"), "-o", str(d / "r.so")], check=True)
    lib = C.CDLL(str(d / "r.so"))

    def call(x, y):
        out = np.empty_like(x)
        p = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
        lib.roots(p(x), p(y), p(out), C.c_uint64(len(x)))
        return out

    return call


@pytest.mark.parametrize("scale", [1e-180, 1e-12, 1.0, 1e12, 1e180])
@pytest.mark.parametrize("off", [-(2.0 ** -23), -(2.0 ** -30), 0.0, 2.0 ** -30, 2.0 ** -23])
def test_root_is_within_an_ulp(roots, scale, off):
    x = scale * np.random.default_rng(7).uniform(0.25, 4.0, size=100000)
    want = np.sqrt(x)
    # half an ulp of the last rounding on each side; what the steps leave is 4e-21
    assert np.all(np.abs(roots(x, (1.0 + off) / want) - want) <= np.spacing(want))


def test_root_of_zero_is_not_a_number(roots):
    assert np.isnan(roots(np.zeros(1), np.array([np.inf])))[0]
