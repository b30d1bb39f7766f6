"""The prior's inputs and outputs at the edges of its pinned buffers (512 KB:
10082 feature rows, 131072 swap targets or matrix entries) and at the largest
multiplier row built in LDS.  Only bytes move and only whole numbers are
drawn, so results must equal, bit for bit, those of calls that stay inside
one buffer; the dense multiplier is compared with the sigmoid of the logits
(fp32, 2e-6 relative: expf against numpy's, then a square)."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import prior as pr

from helpers import log

pytestmark = pytest.mark.gpu

ROWS = 10082   # feature rows of a buffer


def _data(E, seed=1):
    r = np.random.default_rng(seed)
    return r.normal(0, 1, (E, 12)).astype(np.float32), (r.random(E) < 0.1).astype(np.float32)


@pytest.mark.parametrize("E", [1, 15, ROWS - 1, ROWS, ROWS + 1, 2 * ROWS + 1, 40000])
def test_rows_of_every_buffer_arrive(E):
    log(f"prior rows E={E}")
    f, y = _data(E)
    with pr.PriorNet(3) as net:
        whole = net.forward(f)
        parts = np.concatenate([net.forward(f[a:a + 5000]) for a in range(0, E, 5000)])
        np.testing.assert_array_equal(whole, parts)
        # the labels: with weight 1 the loss is the mean over all rows
        _, loss = net.gradient(f, y, 1.0)
        z = whole.astype(np.float64)
        ref = np.mean(np.logaddexp(0.0, z) - y * z)
        assert abs(loss - ref) < 1e-4 * abs(ref) + 1e-6   # E fp32 terms, tree sums


@pytest.mark.parametrize("E,batch,epochs", [(2, 16, 2), (100, 32, 3), (ROWS + 5, 4096, 2), (131073, 65536, 1),
                                            (131074, 65536, 2)])
def test_training_takes_the_shuffled_order(E, batch, epochs):
    log(f"prior training order E={E} batch={batch} epochs={epochs}")
    f, y = _data(E, 2)
    mask, s = (1 << 64) - 1, 77
    with pr.PriorNet(5) as net, pr.PriorNet(5) as step:
        net.train(f, y, epochs=epochs, batch=batch, lr=1e-3, lr_final=1e-3, pos_weight=3.0, shuffle_seed=77)
        for _ in range(epochs):
            perm = list(range(E))
            for i in range(E - 1, 0, -1):
                s = (s + 0x9E3779B97F4A7C15) & mask
                z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
                z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
                j = (z ^ (z >> 31)) % (i + 1)
                perm[i], perm[j] = perm[j], perm[i]
            for b in range(0, E, batch):
                at = np.array(perm[b:b + batch])
                g, _ = step.gradient(f[at], y[at], 3.0)
                step.adam_step(g, 1e-3)
        np.testing.assert_array_equal(net.params(), step.params())


@pytest.mark.parametrize("n,k", [(2, 1), (17, 16), (361, 8), (363, 16), (512, 12), (725, 16), (4096, 4), (4097, 4)])
def test_multiplier_rows(n, k):
    log(f"prior multiplier n={n} k={k}")
    r = np.random.default_rng(n)
    xy = r.integers(0, 1001, size=(n, 2)).astype(np.float64)
    dem = np.concatenate([[0], r.integers(1, 50, size=n - 1)]).astype(np.int32)
    inst = ca.Instance(n=n, x=xy[:, 0].copy(), y=xy[:, 1].copy(), demand=dem, capacity=500,
                       dist=np.hypot(xy[:, None, 0] - xy[None, :, 0], xy[:, None, 1] - xy[None, :, 1]).astype(np.float32))
    # any lists without repeats will do, a column more than is used
    start = r.integers(1, n, size=n)
    nn = ((np.arange(n)[:, None] + 1 + (start[:, None] + np.arange(min(k + 1, n - 1))) % max(n - 1, 1)) % n).astype(np.int32)
    with pr.PriorNet(9) as net:
        got = net.build(inst, nn, k, exponent=2.0, floor=0.05)
        logits = net.forward(pr.features(inst, nn, k)).astype(np.float64).reshape(n, k)
    ref = np.full((n, n), np.float32(0.05) * np.float32(0.05), np.float32)
    np.put_along_axis(ref, nn[:, :k], ((1.0 / (1.0 + np.exp(-logits))) ** 2).astype(np.float32), 1)
    np.testing.assert_allclose(got, ref, rtol=2e-6)
