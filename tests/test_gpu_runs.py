"""A call of n steps (captured runs of 64, 16, 8, 4 and 2, the last odd step
eager) against n calls of one step: the same bits."""
import numpy as np
import pytest

from alya_sma_amd import problems
from alya_sma_amd.solid import Solidz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsteps", [3, 4, 6, 8, 13, 15, 95])
@pytest.mark.parametrize("scheme", [0, 1])
def test_runs_equal_single_steps(scheme, nsteps):
    print("runs of", nsteps, "steps, scheme", scheme, flush=True)
    prob = problems.bar_problem(8, 3, 3, 8.0, 3.0, 3.0, nsteps=200)
    dt = prob["run"]["dt"]
    with Solidz(prob) as a, Solidz(prob) as b:
        for _ in range(2):   # the second call replays the runs
            a.step(dt, nsteps=nsteps, scheme=scheme)
            for _ in range(nsteps):
                b.step(dt, nsteps=1, scheme=scheme)
            for f in ("u", "v", "a", "fint", "sdv", "time"):
                np.testing.assert_array_equal(a.get(f), b.get(f), err_msg=f)
