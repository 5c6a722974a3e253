"""Launches that carry one loading function in the forms of the element kernel
that keep the general code (stored stresses, Rayleigh damping, the surrogate's
prepass and step, other workgroup sizes): the history's second and third array
are then one, and every result has the bits of launches that carry both.  A
negative zero in one point's F_SA is unequal in its bits alone."""
import numpy as np
import pytest

from alya_sma_amd import problems
from alya_sma_amd.solid import Solidz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("form", ["plain", "store", "damped", "store+damped"])
def test_one_loading_function_in_every_form(form, mode):
    print("one loading function", form, mode, flush=True)
    prob = problems.bar_problem()
    dt = prob["run"]["dt"]
    net = None
    if mode == 2:
        from alya_sma_amd import surrogate as S
        net = S.load_default()
        assert net is not None
    with Solidz(prob) as d:
        d.step(dt, nsteps=300)
        st = {f: d.get(f) for f in ("u", "v", "a", "sdv", "time")}
    with Solidz(prob) as one, Solidz(prob) as both:
        still = np.argwhere((st["sdv"] == 0.0).all(axis=2))
        if not len(still):                       # a point whose F is 0, so that -0 equals it
            still = np.array([[0, 0]])
            st["sdv"][0, 0] = 0.0
        for d in (one, both):
            for f, v in st.items():
                v = v.copy()
                if f == "sdv" and d is both:
                    v[tuple(still[0]) + (2,)] = -0.0
                d.set(f, v)
            if "damped" in form:
                d.set_damping(np.array([[1.0e5, 1.0e-9]]))
            if "store" in form:
                d.set_store(True)
            if net is not None:
                d.set_surrogate(net, 1e-4)
            d.set_mode(mode)
            d.step(dt, nsteps=37)
        for f in ("u", "v", "a", "fint", "sdv") + (("stress", "pk1") if "store" in form else ()):
            np.testing.assert_array_equal(one.get(f), both.get(f), err_msg=f)
        assert (one.get("sdv")[..., 0] > 0).any()
        assert one.counters() == both.counters()
    if net is not None:
        net.close()
