"""Scalar functions of the device header, compiled for the host (the hardware
estimates replaced by library ones, the rest the same): J^(-2/3) and the square
root with its reciprocal, over the whole range of doubles and at its ends.

Bounds: two Newton steps on a 24-bit estimate leave the rounding of the last
one, 3 ulps on the squared power and 2 on the root (2 more on the power, for the
step's own factors); scaling by powers of two is exact."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
SRC = r'''
#include "sma_law.hpp"
#include <cstdio>
int main() {
  double x;
  while (fread(&x, 8, 1, stdin) == 1) {
    double o[3] = {sma::pow_m23(x), 0, 0};
    sma::sqrt_rsqrt64(x, o[1], o[2]);
    fwrite(o, 8, 3, stdout);
  }
  return 0;
}
'''


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("scalar")
    (d / "s.cpp").write_text(SRC)
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17",
                    "-I" + os.path.join(ROOT, "alya_sma_amd", "csrc"), str(d / "s.cpp"), "-o",
                    str(d / "s")], check=True, capture_output=True)

    def run(x):
        o = subprocess.run([str(d / "s")], input=np.ascontiguousarray(x, np.float64).tobytes(),
                           capture_output=True, check=True).stdout
        return np.frombuffer(o).reshape(-1, 3).T
    return run


def test_values_over_the_range(prog):
    r = np.random.default_rng(1)
    x = np.concatenate([np.exp2(r.uniform(-1020, 1020, 20000)), 1.0 + 0.1 * r.normal(size=5000),
                        [2.0 ** -100, 2.0 ** 100, np.nextafter(2.0 ** -100, 0), np.nextafter(2.0 ** 100, 4.0 ** 100),
                         1e-290, np.nextafter(1e-290, 0), 5e-324, 1e-310, np.finfo(float).max]])
    x = x[x > 0]
    p, s, i = prog(x)
    X = x.astype(np.longdouble)
    want = [X ** (np.longdouble(-2) / 3), np.sqrt(X), 1 / np.sqrt(X)]
    for got, w, ulps in zip((p, s, i), want, (5, 2, 2)):
        assert np.max(np.abs((got - w) / w)) <= ulps * 2.0 ** -52


def test_ends(prog):
    x = np.array([0.0, -0.0, -1.0, np.inf, np.nan])
    p, s, i = prog(x)
    np.testing.assert_array_equal(p, [np.inf, np.inf, np.nan, 0.0, np.nan])
    assert s[0] == 0.0 and i[0] == 0.0 and s[1] == 0.0 and i[1] == 0.0
    assert np.isnan(s[2]) and i[2] == 0.0 and np.isnan(s[4]) and i[4] == 0.0
