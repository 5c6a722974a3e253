"""Element launches that carry one loading function for both branches (as long
as F_AS and F_SA are equal) against launches that carry both: the same bits,
whatever the assembly, law mix and precision, and through a set history.  A
negative zero in one point's F_SA is unequal in its bits alone, so it keeps
the second handle on the launches with both."""
import numpy as np
import pytest

from alya_sma_amd import problems
from alya_sma_amd.solid import Solidz

pytestmark = pytest.mark.gpu
FIELDS = ("u", "v", "a", "fint", "sdv")


@pytest.mark.parametrize("assembly", ["gather", "scatter"])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("kind", ["bar", "tube"])
def test_one_loading_function_carries_both(kind, mode, assembly):
    print("one loading function", kind, mode, assembly, flush=True)
    prob = (problems.bar_problem(9, 3, 3, 9.0, 3.0, 3.0, nsteps=400) if kind == "bar"
            else problems.cylinder_problem(ntheta=16, nz=6, nr_tube=2, nr_tissue=3, nsteps=400))
    dt = prob["run"]["dt"]
    neo = np.zeros(len(prob["lnods"]), bool)
    if kind == "tube":
        neo = np.asarray(prob["law_of_mat"])[np.asarray(prob["mat_of_elem"])] == problems.LAW_NEOHOOKEAN
    with Solidz(prob) as one, Solidz(prob) as both:
        h = one.get("sdv")
        h[neo] = np.random.default_rng(1).normal(size=h[neo].shape)   # neither read nor written
        hb = h.copy()
        sma = np.flatnonzero(~neo)
        assert np.all(h[sma] == 0.0)
        hb[sma[len(sma) // 2], 5, 2] = -0.0
        one.set("sdv", h)
        both.set("sdv", hb)
        for d in (one, both):
            d.set_mode(mode)
            d.set_assembly(assembly)
            d.step(dt, nsteps=330)
        for f in FIELDS:
            np.testing.assert_array_equal(one.get(f), both.get(f), err_msg=f)
        assert np.any(one.get("sdv")[sma, :, 0] > 0)
        # a history with unequal values ends the short form, an equal one starts it
        h = one.get("sdv")
        hb = h.copy()
        hb[sma, :, 2] *= 1.0 + 1e-3 * np.random.default_rng(2).uniform(size=hb[sma, :, 2].shape)
        one.set("sdv", hb)
        both.set("sdv", hb)
        for d in (one, both):
            d.step(dt, nsteps=21)
        for f in FIELDS:
            np.testing.assert_array_equal(one.get(f), both.get(f), err_msg=f)
        back = both.get("sdv")
        one.set("sdv", back)
        np.testing.assert_array_equal(one.get("sdv"), back)
