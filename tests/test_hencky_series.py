"""The FP64 Hencky strain's series in the invariants of Z (sma::hencky_fp64;
hencky_fp32 beside it, both compiled for the host from the device header) against the same
logarithm in extended precision by products of tensors: strains from 1e-9 to
the series' limit, equal principal values, and strains at every border between
term counts.  Bounds: 32 roundings of the working precision, relative to |E|
(~20 dependent operations lead to a component, the trace sums three)."""
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
  double H[9];
  while (fread(H, 8, 9, stdin) == 9) {
    float Hf[9];
    for (int i = 0; i < 9; ++i) Hf[i] = (float)H[i];
    const sma::Hencky64 a = sma::hencky_fp64(H);
    const sma::Hencky32 b = sma::hencky_fp32(Hf);
    double o[18] = {a.theta, a.e_n, (double)a.ok}, *p = o + 9;
    p[0] = b.theta; p[1] = b.e_n; p[2] = (double)b.ok;
    for (int i = 0; i < 6; ++i) { o[3 + i] = a.ed[i]; p[3 + i] = b.ed[i]; }
    fwrite(o, 8, 18, stdout);
  }
  return 0;
}
'''
L = np.longdouble


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("hencky")
    (d / "h.cpp").write_text(SRC)
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17",
                    "-I" + os.path.join(ROOT, "alya_sma_amd", "csrc"), str(d / "h.cpp"), "-o",
                    str(d / "h")], check=True, capture_output=True)
    return str(d / "h")


def _mm(A, B):
    return (A[:, :, :, None] * B[:, None, :, :]).sum(2)


def _exact(H):
    """theta, |e'|, e' (00, 01, 02, 11, 12, 22) and |Z|_F^2 in extended precision."""
    H = H.astype(L)
    eye = np.eye(3, dtype=L)
    C = H + H.transpose(0, 2, 1) + _mm(H, H.transpose(0, 2, 1))
    M = C + 2 * eye
    a = np.zeros_like(M)
    a[:, 0, 0] = M[:, 1, 1] * M[:, 2, 2] - M[:, 1, 2] ** 2
    a[:, 1, 1] = M[:, 0, 0] * M[:, 2, 2] - M[:, 0, 2] ** 2
    a[:, 2, 2] = M[:, 0, 0] * M[:, 1, 1] - M[:, 0, 1] ** 2
    a[:, 0, 1] = a[:, 1, 0] = M[:, 0, 2] * M[:, 1, 2] - M[:, 0, 1] * M[:, 2, 2]
    a[:, 0, 2] = a[:, 2, 0] = M[:, 0, 1] * M[:, 1, 2] - M[:, 0, 2] * M[:, 1, 1]
    a[:, 1, 2] = a[:, 2, 1] = M[:, 0, 1] * M[:, 0, 2] - M[:, 0, 0] * M[:, 1, 2]
    det = M[:, 0, 0] * a[:, 0, 0] + M[:, 0, 1] * a[:, 0, 1] + M[:, 0, 2] * a[:, 0, 2]
    Z = _mm(C, a) / det[:, None, None]
    W = _mm(Z, Z)
    T, E = Z.copy(), Z.copy()
    for k in range(1, 80):
        T = _mm(T, W)
        E = E + T / (2 * k + 1)
    th = E[:, 0, 0] + E[:, 1, 1] + E[:, 2, 2]
    D = E - th[:, None, None] / 3 * eye
    en = np.sqrt((D * D).sum((1, 2)))
    ed = np.stack([D[:, 0, 0], D[:, 0, 1], D[:, 0, 2], D[:, 1, 1], D[:, 1, 2], D[:, 2, 2]], axis=1)
    return th, en, ed, W[:, 0, 0] + W[:, 1, 1] + W[:, 2, 2]


def _strains():
    """F - I, float32 values: random gradients of all sizes, pure dilatations
    and uniaxial stretches (equal principal values), and gradients scaled onto
    each border of |Z|_F^2 between term counts, a little below and above."""
    rng = np.random.default_rng(3)
    H = [s * rng.normal(size=(200, 3, 3)) for s in (1e-9, 1e-5, 1e-3, 5e-3, 0.02, 0.05, 0.1, 0.15)]
    H.append(rng.uniform(-0.2, 0.2, (100, 1, 1)) * np.eye(3))
    H.append(rng.uniform(-0.2, 0.2, (100, 1, 1)) * np.diag([1.0, -0.33, -0.33]))
    H = [h.astype(np.float32).astype(np.float64) for h in H]
    border = [1.4949e-04, 9.0589e-04, 2.9934e-03, 7.0039e-03, 1.3216e-02, 2.1619e-02, 4.4078e-02,
              1.1898e-01, 2.2961e-01, 0.359, 7.3e-3, 2.6e-2, 5.2e-2, 8.4e-2, 0.115, 0.17, 0.22, 0.28]
    for b in border:
        for f in (0.999, 1.001):
            h = rng.normal(size=(8, 3, 3)) * np.sqrt(b) * 0.3
            for _ in range(60):
                z = _exact(h)[3].astype(float)
                h = h * np.clip(np.sqrt(f * b / z), 0.7, 1.4)[:, None, None]
            H.append(h.astype(np.float32).astype(np.float64))
    return np.concatenate(H)


def test_series_against_extended_precision(prog):
    H = _strains()
    out = subprocess.run([prog], input=np.ascontiguousarray(H.transpose(0, 2, 1)).tobytes(),
                         capture_output=True, check=True).stdout
    out = np.frombuffer(out).reshape(-1, 2, 9)
    th, en, ed, zf2 = _exact(H)
    inside = zf2 < 0.3599
    assert inside.sum() > 1500
    size = np.sqrt(th ** 2 / 3 + en ** 2)[inside]
    for p, eps in ((0, 2.0 ** -53), (1, 2.0 ** -24)):
        r = out[inside, p]
        assert np.all(r[:, 2] == 1)
        assert np.max(np.abs(r[:, 0] - th[inside]) / size) < 32 * eps
        assert np.max(np.abs(r[:, 1] - en[inside]) / size) < 32 * eps
        assert np.max(np.abs(r[:, 3:] - ed[inside]) / size[:, None]) < 32 * eps
