"""The order of the gradient's sums, bit for bit.  A batch of a power of two
of edges scales every term by a power of two, so the terms are the gradients
of smaller batches, scaled: single edges for the biases and the last layer,
64 edges (one partial row) for everything."""
import numpy as np
import pytest

from cvrp_aco_ocl_amd import prior
from oracle import prior as P

from helpers import log

pytestmark = pytest.mark.gpu

f32 = np.float32
ROW = 64   # edges of a partial row: four tiles of 16


def edges(E, seed):
    r = np.random.default_rng(seed)
    return r.uniform(0.0, 1.5, (E, 12)).astype(f32), (r.random(E) < 0.2).astype(f32)


def terms(net, f, y):
    g, loss = net.gradient(f, y, 3.0)
    return np.append(g, f32(loss))


def tree(a):
    """Sixteen lanes' butterfly sum (lane 0's)."""
    for o in (1, 2, 4, 8):
        a = a + a[np.arange(16) ^ o]
    return a[0]


@pytest.mark.parametrize("E", [1, 2, 8, 16, 32, 64])
def test_edges_of_a_row(E):
    """Lane r adds edge r of each tile in turn, then the lanes are added."""
    log(f"prior sum order of a row, E={E}")
    f, y = edges(E, E)
    with prior.PriorNet(seed=4) as net:
        g = terms(net, f, y)
        t = np.stack([terms(net, f[e:e + 1], y[e:e + 1]) for e in range(E)])
    scale = f32(1.0) / f32(E)
    cols = np.r_[P.OFF_B1:P.OFF_W2, P.OFF_B2:P.NPARAM + 1]   # biases, last layer, loss
    assert cols[-1] == len(g) - 1
    lanes = np.zeros((16, len(g)), f32)
    for e in range(E):
        lanes[e % 16] += t[e]
    np.testing.assert_array_equal(g[cols], (tree(lanes) * scale)[cols])


@pytest.mark.parametrize("E", [64, 128, 256, 512, 1024, 4096, 16384, 32768, 65536])
def test_rows_of_a_batch(E):
    """Consecutive rows in eight runs, each in order, then the runs."""
    log(f"prior sum order of the rows, E={E}")
    f, y = edges(E, E + 1)
    with prior.PriorNet(seed=4) as net:
        g = terms(net, f, y)
        t = np.stack([terms(net, f[i:i + ROW], y[i:i + ROW]) for i in range(0, E, ROW)]) * f32(ROW / E)
    rows = -(-len(t) // 4) * 4
    run = -(-rows // 8)
    runs = []
    for a in range(0, len(t), run):
        s = np.zeros(len(g), f32)
        for row in t[a:a + run]:
            s = s + row
        runs.append(s)
    s = runs[0]
    for q in runs[1:]:
        s = s + q
    np.testing.assert_array_equal(g, s)
