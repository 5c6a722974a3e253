"""sma160_eval's staging (chunks of points through slots of pinned memory that
the kernel reads and writes) against sma160_eval_device on the same points: the
same kernel, so the same bits, at the edges of chunks and slots, with each
optional array left out, in place, with overlapping arrays and from several
threads."""
import threading

import numpy as np
import pytest

from alya_sma_amd._lib import check, lib
from alya_sma_amd.device import DeviceArray, synchronize
from alya_sma_amd.problems import NITINOL

pytestmark = pytest.mark.gpu
CHUNK, SLOTS = 6144, 4


def _a(x):
    return None if x is None else x.__array_interface__["data"][0]


def _points(n, nmat, seed):
    r = np.random.default_rng(seed)
    props = np.tile(NITINOL, (nmat, 1))
    props[:, 0] *= r.uniform(0.9, 1.1, nmat)
    F = 0.01 * r.normal(size=(9, n))
    F[[0, 4, 8]] += 1.0
    sdv = np.stack([r.uniform(size=n), 300 * r.uniform(size=n), 300 * r.uniform(size=n)])
    return props, F, sdv, r.integers(0, nmat, n).astype(np.int32), 60000.0 * r.uniform(0.98, 1.02, n)


def _device(props, F, sdv, mat, E, prec):
    n = F.shape[1]
    d = [None if x is None else DeviceArray.from_host(x) for x in (props, mat, E, F, sdv)]
    sn, S, fl = DeviceArray((3, n), np.float64), DeviceArray((9, n), np.float64), DeviceArray((n,), np.uint32)
    p = [None if x is None else x.ptr for x in d]
    check(lib().sma160_eval_device(n, len(props), p[0], p[1], p[2], p[3], None, p[4], sn.ptr, S.ptr,
                                   fl.ptr, prec, None), "sma160_eval_device")
    synchronize()
    return sn.to_host(), S.to_host(), fl.to_host()


def _host(props, F, sdv, mat, E, prec, sn, S, fl):
    check(lib().sma160_eval(F.shape[1], len(props), _a(props), _a(mat), _a(E), _a(F), None, _a(sdv),
                            _a(sn), _a(S), _a(fl), prec), "sma160_eval")


@pytest.mark.parametrize("n", [1, 63, CHUNK - 1, CHUNK, CHUNK + 1, SLOTS * CHUNK, SLOTS * CHUNK + 1, 130 * 6100])
def test_chunks_match_the_device_call(n):
    print(f"law host call, {n} points", flush=True)
    props, F, sdv, mat, E = _points(n, 3, n)
    for m, e, prec, flags in ((mat, E, 0, True), (None, E, 0, False), (mat, None, 1, True)):
        sn, S, fl = np.empty((3, n)), np.empty((9, n)), np.empty(n, np.uint32) if flags else None
        _host(props, F, sdv, m, e, prec, sn, S, fl)
        sd, Sd, fd = _device(props, F, sdv, m, e, prec)
        np.testing.assert_array_equal(sn, sd)
        np.testing.assert_array_equal(S, Sd)
        if flags:
            np.testing.assert_array_equal(fl, fd)


def test_in_place_and_overlapping_arrays():
    n = 3 * CHUNK + 17
    props, F, sdv, mat, E = _points(n, 3, 5)
    sd, Sd, _ = _device(props, F, sdv, mat, E, 0)
    f, s = F.copy(), sdv.copy()
    _host(props, f, s, mat, E, 0, s, f, None)
    np.testing.assert_array_equal(s, sd)
    np.testing.assert_array_equal(f, Sd)
    for shift in (-1000, 1000):   # the history out overlaps the history in, elsewhere
        buf = np.zeros(3 * n + 2000)
        old, new = buf[1000:1000 + 3 * n].reshape(3, n), buf[1000 + shift:1000 + shift + 3 * n].reshape(3, n)
        old[:] = sdv
        S = np.empty((9, n))
        _host(props, F, old, mat, E, 0, new, S, None)
        np.testing.assert_array_equal(new, sd)
        np.testing.assert_array_equal(S, Sd)


def test_calls_from_several_threads():
    cases = [_points(n, 2, n) for n in (8, 100, CHUNK + 3, 2 * CHUNK, 8, 30000)]
    want = [_device(*c, 0) for c in cases]
    bad = []

    def work(c, w):
        for _ in range(5):
            n = c[1].shape[1]
            sn, S, fl = np.empty((3, n)), np.empty((9, n)), np.empty(n, np.uint32)
            _host(*c, 0, sn, S, fl)
            if not (np.array_equal(sn, w[0]) and np.array_equal(S, w[1]) and np.array_equal(fl, w[2])):
                bad.append(n)

    ts = [threading.Thread(target=work, args=x) for x in zip(cases, want)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
