"""root8 of the state rates, x**0.125 for x >= 1, against 60-digit arithmetic:
compiled for the host from the kernels' own header (the square root and the
fused multiply-add round alike there and on the device).

Half an ulp for the last sum, and for the corrections, which are at most 1.04
ulp, their own rounding (under ten operations, 2^-53 each) and what the
first-order residuals leave out (2^-53 of them): below 0.5001 ulp.  The points
are random over the whole range, every binade's ends, and the neighbourhood of
16, where plain square roots are off by more than an ulp.
"""
import ctypes
import math
import os
import subprocess
from decimal import Decimal, getcontext

import numpy as np
import pytest

from conftest import ROOT

SRC = """
#include "fdm_physics.hpp"
extern "C" void roots(const double* x, double* y, int n) {
  for (int k = 0; k < n; k++) y[k] = fdm::root8(x[k]);
}
"""


@pytest.fixture(scope="module")
def roots(tmp_path_factory):
    d = tmp_path_factory.mktemp("root8")
    src, lib = d / "root8.hip", d / "libroot8.so"
    src.write_text(SRC)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-O2", "-std=c++17", "-fPIC",
                    "-shared", "-ffp-contract=off", "-I", os.path.join(ROOT, "fdmap_github_amd", "csrc"), "-o",
                    str(lib), str(src)], check=True, timeout=300)
    fn = ctypes.CDLL(str(lib)).roots

    def call(x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        y = np.empty_like(x)
        fn(x.ctypes.data_as(ctypes.c_void_p), y.ctypes.data_as(ctypes.c_void_p), ctypes.c_int(x.size))
        return y

    return call


def test_error(roots):
    getcontext().prec = 60
    rng = np.random.default_rng(8)
    two = 2.0 ** np.arange(0, 1024)
    x = np.concatenate([[16.08906214441935, 16.672113509682728], 16.0 * (1.0 + 0.1 * rng.random(3000)),
                        1.0 + rng.random(3000), 10.0 ** rng.uniform(0, 308, 3000), two, np.nextafter(two, np.inf),
                        np.nextafter(two[1:], 0.0), [np.finfo(float).max]])
    worst = max(abs((Decimal(float(v)) - Decimal(float(u)).sqrt().sqrt().sqrt()) / Decimal(math.ulp(v)))
                for u, v in zip(x, roots(x)))
    assert worst < Decimal("0.5001"), worst


def test_ends(roots):
    y = roots([1.0, 256.0, np.inf, np.nan])
    assert y[0] == 1.0 and y[1] == 2.0 and y[2] == np.inf and np.isnan(y[3])
