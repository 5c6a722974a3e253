"""The point-wise FP64 law at singular deformation gradients: where the reference
divides a finite Kirchhoff stress by det F = 0, its infinite stresses come back,
with their signs.  F of small integers over 8, rank 2, so that det F is an exact
zero in any order of operations; the eigenvalue of b that should be zero is
rounding, positive or not (then NaN), and the oracle says which."""
import numpy as np
import pytest

from alya_sma_amd.device import DeviceArray, synchronize
from alya_sma_amd.problems import NITINOL
from alya_sma_amd.solid import eval_sld_stress_model_160, eval_sld_stress_model_160_device
from conftest import soa
from oracle import oracle_py as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 4000])
def test_singular_gradients_give_the_references_infinities(n):
    print("singular gradients", n, flush=True)
    r = np.random.default_rng(0)
    F = (r.integers(-4, 5, (n, 3, 2)) @ r.integers(-4, 5, (n, 2, 3))) / 8.0
    F = np.ascontiguousarray(soa(F))
    sdv = np.ascontiguousarray(np.tile([[0.2], [100.0], [100.0]], (1, n)))
    _, So, fo = O.sm160_eval(NITINOL[None], F, sdv)
    inf = np.isinf(So).all(axis=0)
    assert inf.any()
    _, S, fl = eval_sld_stress_model_160(NITINOL[None], F, sdv)
    np.testing.assert_array_equal(S[:, inf], So[:, inf])
    np.testing.assert_array_equal(fl[inf], fo[inf])
    d = [DeviceArray.from_host(x) for x in (NITINOL[None], F, sdv)]
    sn, Sd, fd = DeviceArray((3, n), np.float64), DeviceArray((9, n), np.float64), DeviceArray((n,), np.uint32)
    eval_sld_stress_model_160_device(n, 1, d[0].ptr, d[1].ptr, d[2].ptr, sn.ptr, Sd.ptr, flags_ptr=fd.ptr)
    synchronize()
    np.testing.assert_array_equal(Sd.to_host(), S)
