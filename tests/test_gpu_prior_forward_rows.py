"""Logits of more edges than one copy of features moves (131072 rows): one
row short of it, one past it, and two copies and a row, on a network that has
already been used for less and for more.  Rows are independent, so every part
must equal, bit for bit, the same rows asked for alone."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca

from helpers import log

pytestmark = pytest.mark.gpu

ROWS = 131072


@pytest.mark.parametrize("first", [5, 2 * ROWS + 100])
@pytest.mark.parametrize("E", [1, ROWS - 1, ROWS, ROWS + 1, 2 * ROWS + 1])
def test_logits_of_several_copies(E, first):
    log(f"forward rows E={E} after {first}")
    f = np.random.default_rng(E).normal(0, 1, (E, 12)).astype(np.float32)
    with ca.prior.PriorNet(3) as net:
        net.forward(np.ones((first, 12), np.float32))
        whole = net.forward(f)
        parts = np.concatenate([net.forward(f[a:a + 30001]) for a in range(0, E, 30001)])
        np.testing.assert_array_equal(whole, parts)
        np.testing.assert_array_equal(net.forward(f), whole)
