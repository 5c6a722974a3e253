"""sma160_eval with arrays that share memory, at sizes of several chunks: all
inputs are read before the first output is stored, and the history, the stresses
and the flags are stored whole and in this order, so the last one stored is right
wherever it lies."""
import numpy as np
import pytest

from alya_sma_amd._lib import check, lib
from alya_sma_amd.problems import NITINOL

pytestmark = pytest.mark.gpu
CHUNK = 6144


def _at(x, byte=0):
    return x.__array_interface__["data"][0] + byte


def _call(n, F, sdv, sn, S, fl):
    check(lib().sma160_eval(n, 1, _at(PROPS), None, None, F, None, sdv, sn, S, fl, 0), "sma160_eval")


PROPS = np.ascontiguousarray(NITINOL[None], dtype=np.float64)


@pytest.fixture(scope="module", params=[CHUNK, CHUNK + 1, 5 * CHUNK + 17])
def points(request):
    n = request.param
    r = np.random.default_rng(n)
    F = 0.01 * r.normal(size=(9, n))
    F[[0, 4, 8]] += 1.0
    sdv = np.stack([r.uniform(size=n), 300 * r.uniform(size=n), 300 * r.uniform(size=n)])
    sn, S, fl = np.empty((3, n)), np.empty((9, n)), np.empty(n, np.uint32)
    _call(n, _at(F), _at(sdv), _at(sn), _at(S), _at(fl))
    return n, F, sdv, sn, S, fl


@pytest.mark.parametrize("where", ["F", "sdv_old"])
def test_flags_over_an_input(points, where):
    n, F, sdv, sn0, S0, fl0 = points
    print("flags over", where, n, flush=True)
    F, sdv, sn, S = F.copy(), sdv.copy(), np.empty((3, n)), np.empty((9, n))
    buf = F if where == "F" else sdv
    _call(n, _at(F), _at(sdv), _at(sn), _at(S), _at(buf))
    np.testing.assert_array_equal(buf.reshape(-1).view(np.uint32)[:n], fl0)
    np.testing.assert_array_equal(sn, sn0)
    np.testing.assert_array_equal(S, S0)


@pytest.mark.parametrize("shift", [0, 8 * 777])
def test_outputs_over_each_other(points, shift):
    n, F, sdv, sn0, S0, fl0 = points
    print("outputs over each other", n, shift, flush=True)
    buf = np.empty(9 * n + 1000)       # the stresses over the history
    fl = np.empty(n, np.uint32)
    _call(n, _at(F), _at(sdv), _at(buf, shift), _at(buf), _at(fl))
    np.testing.assert_array_equal(buf[:9 * n].reshape(9, n), S0)
    np.testing.assert_array_equal(fl, fl0)
    sn = np.empty((3, n))              # the flags over the stresses
    _call(n, _at(F), _at(sdv), _at(sn), _at(buf), _at(buf, shift))
    np.testing.assert_array_equal(buf.view(np.uint32)[shift // 4:shift // 4 + n], fl0)
    np.testing.assert_array_equal(sn, sn0)


def test_outputs_in_place(points):
    n, F, sdv, sn0, S0, _ = points
    print("in place", n, flush=True)
    F, sdv = F.copy(), sdv.copy()
    _call(n, _at(F), _at(sdv), _at(sdv), _at(F), None)
    np.testing.assert_array_equal(sdv, sn0)
    np.testing.assert_array_equal(F, S0)
    # the stresses over the old history, the new history over F
    n, F, sdv, sn0, S0, _ = points
    buf, f = np.empty(9 * n), F.copy()
    buf[:3 * n] = sdv.reshape(-1)
    _call(n, _at(f), _at(buf), _at(f), _at(buf), None)
    np.testing.assert_array_equal(buf.reshape(9, n), S0)
    np.testing.assert_array_equal(f.reshape(-1)[:3 * n], sn0.reshape(-1))
