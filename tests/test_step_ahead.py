"""The rule by which FGMRES launches an Arnoldi step before it has read the flags of the
step before (helmholtz.jl_amd/csrc/hh_ahead.h), compiled with g++ and driven as the
solver drives it over sequences of residual estimates: no step is launched past the end
of a solve that converges at a steady rate or in one step, and only the last few steps of
a long one are waited for.  CPU only."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "helmholtz.jl_amd", "csrc", "hh_ahead.h")

# est[k]: the estimate after step k of the solve; restart cycles of K steps, each beginning
# with the last one's estimate.  out: steps launched past the end, steps waited for.
SRC = r"""
#include "%s"
extern "C" void drive(int n, const double* est, int K, double tol, int* out) {
  hh::StepAhead rule(tol);
  out[0] = out[1] = 0;
  int k0 = 0;
  for (;;) {
    if (k0 > 0) rule.restart(est[k0 - 1]);
    int known = 0;
    bool end = false;
    for (int j = 0; j < K && !end; ++j) {  // step j is launched here
      if (k0 + j >= n) { ++out[0]; return; }  // it was past the end, and step j - 1's flags say so
      for (; known < j && !end; ++known) {
        rule.step(est[k0 + known]);
        end = !(est[k0 + known] > tol);
      }
      if (end) { ++out[0]; return; }
      if (j + 1 < K && rule.may_end()) {
        ++out[1];
        rule.step(est[k0 + known]);
        end = !(est[k0 + known] > tol);
        ++known;
      }
    }
    for (; k0 + known < n && known < K; ++known) {
      rule.step(est[k0 + known]);
      end = end || !(est[k0 + known] > tol);
    }
    k0 += known;
    if (end || k0 >= n) return;
  }
}
"""


@pytest.fixture(scope="module")
def drive(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("ahead")
    src, lib = d / "a.cpp", d / "a.so"
    src.write_text(SRC % HEADER)
    subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    f = C.CDLL(str(lib)).drive

    def go(est, K, tol):
        e = np.ascontiguousarray(est, dtype=np.float64)
        out = (C.c_int * 2)()
        f(len(e), e.ctypes.data_as(C.POINTER(C.c_double)), K, C.c_double(tol), out)
        return out[0], out[1]
    return go


def series(rate, tol):
    """The steady estimates up to the first that meets the tolerance (0.1**3 does not meet 1e-3)."""
    e = rate ** np.arange(1, 1200)
    return e[: int(np.argmax(e <= tol)) + 1]


@pytest.mark.parametrize("K", [2, 5, 10, 32])
@pytest.mark.parametrize("tol", [0.9, 0.5, 1e-1, 1e-3, 1e-6, 1e-12])
@pytest.mark.parametrize("rate", [1e-15, 1e-3, 0.1, 0.5, 0.87, 0.97])
def test_steady(drive, rate, tol, K):
    past, waited = drive(series(rate, tol), K, tol)
    assert past == 0
    assert waited <= 3  # the first step and the end


@pytest.mark.parametrize("K", [5, 10])
@pytest.mark.parametrize("seed", range(20))
def test_uneven(drive, seed, K):
    """Rates that wander by a factor of 30 in their logarithm about a mean of 0.87: at
    most one step past the end, and a tenth of the steps waited for."""
    rng = np.random.default_rng(seed)
    e = np.cumprod(np.exp(np.log(0.87) * np.exp(rng.normal(0.0, 1.1, 400))))
    e = e[: int(np.argmax(e <= 1e-6)) + 1]
    past, waited = drive(e, K, 1e-6)
    assert past <= 1
    assert waited <= 3 + len(e) // 10


def test_not_a_number(drive):
    """A non-finite estimate ends the solve by its flag; the rule only has to return."""
    assert drive([0.5, float("nan")], 10, 1e-6)[0] <= 1
