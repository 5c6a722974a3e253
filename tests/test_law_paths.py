"""The point-wise FP64 law (sma::law_point, series strain where it applies)
against its spectral form at the same points, both compiled for the host from
the device header: strains from 1e-9 to stretches beyond the series, rotations,
the unit deformation, equal principal values, singular, reflecting and
non-finite F, every branch of the return map, materials in Pa (whose residuals
need the reference's iteration).

Bounds: both forms carry rounding of about 1e-16 into the strain, the spectral
form ~30 operations of it (eigenvalues, root, power, logarithm), so the
loading functions agree to 64 eps (2G + 9 |alfa| K); the return map divides that
by its slope, 2G eL + G_1 and more, so xS to 64 eps (1 + 9 |alfa| K / 2G) / eL
and the stress, through the direction e'/|e'| of a transformed point, to
64 eps (2G (1 + eL xS / |e'|) + 3K) times the pull-back.  Flags and iteration
counts are equal."""
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle_py as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")

SRC = r'''
#include "sma_law.hpp"
#include <cstdio>
using namespace sma;
int main() {
  double b[30];
  while (fread(b, 8, 30, stdin) == 30) {
    double F[9], Fi[9], tau[6], S[9];
    for (int i = 0; i < 9; ++i) F[i] = b[18 + i];
    const Mat m = make_mat(b, b[0]);
    inv3<double>(F, Fi);
    for (int k = 0; k < 2; ++k) {
      ReturnMap r;
      const Spectral<double> sp = spectral_fp64(F);
      if (k == 0) {
        r = law_point(m, F, b[27], b[28], b[29], tau);
      } else {
        r = return_map(m, sp.theta, sp.e_n, b[27], b[28], b[29]);
        if (!sp.eig_ok) r.flags |= FLAG_EIGEN_FAIL;
        kirchhoff<double>(m, sp, r.xS, tau);
      }
      pk2<double>(Fi, tau, S);
      double o[14] = {r.xS, r.F_AS, r.F_SA, (double)r.flags, sp.e_n};
      for (int i = 0; i < 9; ++i) o[5 + i] = S[i];
      fwrite(o, 8, 14, stdout);
    }
  }
  return 0;
}
'''
NITINOL = np.array([60000, 0.33, 0.05, 400, 500, 0, 0, 0, 0, 250, 150, 0, 0, 0, 0, 1, 1, 0.0])
EPS = 2.0 ** -52


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("law")
    (d / "l.cpp").write_text(SRC)
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17",
                    "-I" + os.path.join(ROOT, "alya_sma_amd", "csrc"), str(d / "l.cpp"), "-o",
                    str(d / "l")], check=True, capture_output=True)

    def run(P, F, sdv):
        b = np.concatenate([P, F.transpose(0, 2, 1).reshape(-1, 9), sdv], 1)
        o = subprocess.run([str(d / "l")], input=np.ascontiguousarray(b).tobytes(),
                           capture_output=True, check=True).stdout
        o = np.frombuffer(o).reshape(-1, 2, 14)
        return o[:, 0], o[:, 1]
    return run


def _rotations(r, n):
    q, _ = np.linalg.qr(r.normal(size=(n, 3, 3)))
    return q * np.sign(np.linalg.det(q))[:, None, None]


def _compare(P, F, a, b):
    G2 = P[:, 0] / (1 + P[:, 1])
    K = P[:, 0] / (3 * (1 - 2 * P[:, 1]))
    s3, s23 = np.sqrt(1 / 3), np.sqrt(2 / 3)
    alfa = np.abs(s23 * (P[:, 4] - P[:, 3]) / (P[:, 4] + P[:, 3]) * s3) + s3
    np.testing.assert_array_equal(a[:, 3], b[:, 3])
    np.testing.assert_array_equal(np.isfinite(a), np.isfinite(b))
    ok = np.isfinite(b).all(1)
    a, b, F, G2, K, alfa, eL = a[ok], b[ok], F[ok], G2[ok], K[ok], alfa[ok], P[ok, 2]
    rel = 1 + 9 * alfa * K / G2
    assert (np.abs(a[:, 0] - b[:, 0]) <= 64 * EPS * rel / eL).all()
    big = np.maximum(np.abs(b[:, 1]), G2 * rel)
    assert (np.abs(a[:, 1:3] - b[:, 1:3]) <= 64 * EPS * 4 * big[:, None]).all()
    en = np.maximum(b[:, 4], 1e-300)
    pull = np.linalg.norm(np.linalg.inv(F), axis=(1, 2)) ** 2
    tol = 64 * EPS * (G2 * (1 + eL * b[:, 0] / en) + 3 * K) * rel * pull
    same = (a[:, 5:] == b[:, 5:]).all(1)
    assert (same | (np.abs(a[:, 5:] - b[:, 5:]).max(1) <= tol)).all()


def _points(size, unit, n=4000):
    """Points around a strain, transformed or not, the history near the loading
    functions of the strain; stresses in MPa / unit."""
    r = np.random.default_rng(int(size * 1e9) % 2 ** 31)
    P = np.tile(NITINOL, (n, 1))
    P[:, [0, 3, 4, 9, 10]] *= r.uniform(0.9, 1.1, (n, 5)) * unit
    H = size * r.normal(size=(n, 3, 3))
    en = np.linalg.norm(H + H.transpose(0, 2, 1), axis=(1, 2)) / 2
    G2 = P[:, 0] / (1 + P[:, 1])
    xs = np.where(r.uniform(size=n) < 0.3, 0.0, np.where(r.uniform(size=n) < 0.2, 1.0, r.uniform(size=n)))
    f0 = G2 * (en - P[:, 2] * xs) * r.uniform(0.8, 1.2, n) + r.normal(size=n) * unit
    return P, H, np.stack([xs, f0, f0], 1)


@pytest.mark.parametrize("unit", [1e-3, 1.0, 1e3, 1e6])
@pytest.mark.parametrize("size", [1e-4, 1e-3, 0.01, 0.05])
def test_return_map_ends_as_the_oracle(prog, size, unit):
    """In Pa (unit 1e6) rounding alone exceeds the iteration's tolerance: whether
    and when it ends must still be the reference's."""
    P, H, sdv = _points(size, unit)
    F = np.eye(3) + H
    n = len(F)
    so, S, fl = O.sm160_eval(P, np.ascontiguousarray(F.transpose(0, 2, 1).reshape(n, 9).T),
                             np.ascontiguousarray(sdv.T), mat_of_gp=np.arange(n))
    _, a = prog(P, F, sdv)
    np.testing.assert_array_equal(a[:, 3].astype(int) & 0xff0f, fl.astype(int) & 0xff0f)
    np.testing.assert_allclose(a[:, 0], so[0], rtol=0, atol=1e-12)


@pytest.mark.parametrize("unit", [1.0, 1e6])
@pytest.mark.parametrize("size", [1e-9, 9e-6, 1.1e-5, 1e-4, 1e-3, 0.01, 0.05, 0.2, 0.6])
def test_series_and_spectral_law_agree(prog, size, unit):
    P, H, sdv = _points(size, unit)
    r = np.random.default_rng(3)
    H[:300] = size * r.normal(size=(300, 1, 1)) * np.diag([1.0, -0.35, -0.35])
    H[300:500] = size * r.normal(size=(200, 1, 1)) * np.eye(3)
    F = np.eye(3) + H
    F[500:900] = F[500:900] @ _rotations(r, 400)
    a, b = prog(P, F, sdv)
    _compare(P, F, a, b)


def test_special_deformations(prog):
    F = [np.eye(3), -np.eye(3), np.diag([1.0, 1, -1]), np.diag([1.0, 1, 0]), np.zeros((3, 3)),
         np.diag([3.0, 1, 1]), np.diag([1e200, 1, 1]), np.diag([1e-200, 1, 1]), np.full((3, 3), np.nan),
         np.diag([np.inf, 1, 1]), np.eye(3) + np.nan * np.diag([1.0, 0, 0])]
    F += list(_rotations(np.random.default_rng(1), 20))
    F = np.array(F)
    n = len(F)
    P = np.tile(NITINOL, (n, 1))
    for sdv in ([0, 0, 0], [0.5, 100, 100], [1, 600, 600], [0.2, np.nan, 0], [np.nan, 0, 0], [0.2, np.inf, 0],
                [0.2, -np.inf, np.inf]):
        a, b = prog(P, F, np.tile(np.array(sdv, float), (n, 1)))
        # deviatoric strains of rounding size take the spectral form: the same bits
        np.testing.assert_array_equal(a, b)


def test_underflow_band_keeps_the_references_answer(prog):
    """Shear strains whose fourth powers underflow in the reference's
    Householder step: its NaN, where it gives one, bit for bit otherwise."""
    tiny = 10.0 ** np.arange(-200, -68, 1.5)
    F = np.tile(np.diag([1.02, 0.995, 0.99]), (3 * len(tiny), 1, 1))
    for k, (i, j) in enumerate(((0, 1), (0, 2), (1, 2))):
        F[k * len(tiny):(k + 1) * len(tiny), i, j] = tiny
    n = len(F)
    P = np.tile(NITINOL, (n, 1))
    a, b = prog(P, F, np.tile([0.0, 0.0, 0.0], (n, 1)))
    assert np.isnan(b).any()
    np.testing.assert_array_equal(a, b)
