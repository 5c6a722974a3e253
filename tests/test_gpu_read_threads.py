"""Fields read by several threads at once, and by a thread whose current device
is not the handle's: a read changes nothing of the handle and allocates on no
device, so every reader gets the same values."""
import ctypes as C
import threading

import numpy as np
import pytest

from alya_sma_amd import problems
from alya_sma_amd.device import device_count
from alya_sma_amd.solid import Solidz

pytestmark = pytest.mark.gpu


def _handle():
    """A law-grouped mesh whose stored order is not the caller's."""
    prob = problems.cylinder_problem(ntheta=48, nz=20, nr_tube=2, nr_tissue=4, nsteps=400)
    d = Solidz(prob)
    h = np.random.default_rng(1).normal(size=(d.nelem, 8, 3))
    d.set("sdv", h)
    return d, h


def _read(d, n, before=lambda: None):
    got, err = [None] * n, []
    gate = threading.Barrier(n)

    def work(k):
        try:
            before()
            gate.wait()
            got[k] = d.get("sdv")
        except Exception as e:   # noqa: BLE001
            err.append(e)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(n)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not err
    return got


def test_first_reads_by_several_threads():
    print("first reads by threads", flush=True)
    for _ in range(5):
        d, h = _handle()
        with d:
            for x in _read(d, 8):
                np.testing.assert_array_equal(x, h)


def test_reader_on_another_device():
    if device_count() < 2:
        pytest.skip("one device")
    # the HIP runtime that the library links
    hip = C.CDLL(next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x))
    d, h = _handle()
    with d:
        for x in _read(d, 2, before=lambda: hip.hipSetDevice(1)):
            np.testing.assert_array_equal(x, h)
