"""Hidden units far on the closed side of SiLU, as a diverging run or a set network
can have them: training sees the 0 that inference sees, in the output and in the
gradient, however large the negative pre-activation is.

Tolerances as for ragged batches: the oracle rounds at the same points, so what
remains is a BF16 ulp (2^-8) in a small share of the operands; blocks by norm at
2^-7, the loss at 1e-3."""
import numpy as np
import pytest

from alya_sma_amd.device import DeviceArray
from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


@pytest.mark.filterwarnings("ignore:overflow")
@pytest.mark.parametrize("closed", [-80.0, -90.0, -1e4, -1e30, -3e36, -3e38])
def test_closed_units_in_training(closed):
    from alya_sma_amd.surrogate import Surrogate
    print(f"training with units at {closed}", flush=True)
    rng = np.random.default_rng(2)
    n = 200
    X = rng.normal(size=(n, 16)).astype(np.float32)
    T = rng.normal(size=(n, 12)).astype(np.float32)
    s = Surrogate(seed=5)
    s.set_loss_weights(np.ones(12, np.float32))
    W, b = s.get_params()
    for l in range(4):
        b[128 * l + 3:128 * l + 128:6] = closed
    s.set_params(W, b)
    loss, gW, gb = s.grad(DeviceArray.from_host(X), DeviceArray.from_host(T))
    Y = s.forward(DeviceArray.from_host(X)).to_host()
    s.close()
    Lo, gWo, gbo = M.loss_and_grad(W, b, X, T, emulate=True)
    assert abs(np.sum((Y.astype(float) - T) ** 2) / n - Lo) <= 1e-3 * Lo      # inference
    assert abs(loss - Lo) <= 1e-3 * Lo
    o = ob = 0
    for (nn, kk) in M.SIZES:
        for g, go in ((gW[o:o + nn * kk], gWo[o:o + nn * kk]), (gb[ob:ob + nn], gbo[ob:ob + nn])):
            assert np.linalg.norm(g - go) <= 2.0 ** -7 * np.linalg.norm(go)
        o, ob = o + nn * kk, ob + nn
