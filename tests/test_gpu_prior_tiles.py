"""The prior's gradient where a wave takes more than one tile of 16 edges:
one edge short of every block's first tiles and past them, a last tile of one
edge, the second and the fourth tile per wave and the largest batch.  Against
the oracle, with the bounds of the smaller sizes (bf16 operands on both
sides; the sums differ in order only)."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from oracle import prior as P

from helpers import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [16383, 16384, 16385, 16449, 32768, 32769, 49153, 65535, 65536])
def test_gradient_of_several_tiles_per_wave(E):
    log(f"gradient tiles E={E}")
    r = np.random.default_rng(E)
    f = r.uniform(0.0, 1.5, (E, 12)).astype(np.float32)
    y = (r.random(E) < 0.15).astype(np.float32)
    with ca.prior.PriorNet(seed=9) as net:
        p = net.params()
        g, loss = net.gradient(f, y, 4.0)
        again, _ = net.gradient(f, y, 4.0)
    np.testing.assert_array_equal(g, again)
    gr, lr = P.backward(p, f, y, 4.0)
    assert abs(loss - lr) <= 1e-5 * abs(lr)
    assert np.abs(g - gr).max() <= 2e-3 * np.abs(gr).max()
    for lo, hi in ((P.OFF_W1, P.OFF_B1), (P.OFF_B1, P.OFF_W2), (P.OFF_W2, P.OFF_B2), (P.OFF_B2, P.OFF_W3),
                   (P.OFF_W3, P.OFF_B3)):
        assert np.abs(g[lo:hi] - gr[lo:hi]).max() <= 1e-2 * np.abs(gr[lo:hi]).max() + 1e-9, (lo, hi)
