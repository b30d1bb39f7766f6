"""Training whose epochs draw their swap targets on the host (fewer than 4096
draws) and on the device, on both sides of the line: one epoch, two (the
requests ahead) and more, and twice on one network; and epochs of two buffers
(131072 draws each), whose third and later epochs draw beside the training.  The order is written out here; the batches it gives, taken
one by one with gradient and Adam step, must give the same parameters, bit
for bit."""
import numpy as np
import pytest

from cvrp_aco_ocl_amd import prior as pr

from helpers import log

pytestmark = pytest.mark.gpu

MASK = (1 << 64) - 1


def _orders(E, epochs, seed):
    s = seed
    for _ in range(epochs):
        perm = list(range(E))
        for i in range(E - 1, 0, -1):
            s = (s + 0x9E3779B97F4A7C15) & MASK
            z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & MASK
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK
            j = (z ^ (z >> 31)) % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        yield np.array(perm)


@pytest.mark.parametrize("epochs", [1, 2, 5])
@pytest.mark.parametrize("E", [1, 2, 17, 4096, 4097, 4098])
def test_order_of_small_and_large_epochs(E, epochs):
    log(f"training draws E={E} epochs={epochs}")
    r = np.random.default_rng(E)
    f, y = r.normal(0, 1, (E, 12)).astype(np.float32), (r.random(E) < 0.1).astype(np.float32)
    with pr.PriorNet(5) as net, pr.PriorNet(5) as step:
        for seed in (77, (1 << 64) - 3):
            net.train(f, y, epochs=epochs, batch=1024, lr=1e-3, lr_final=1e-3, pos_weight=3.0, shuffle_seed=seed)
            for perm in _orders(E, epochs, seed):
                for b in range(0, E, 1024):
                    at = perm[b:b + 1024]
                    g, _ = step.gradient(f[at], y[at], 3.0)
                    step.adam_step(g, 1e-3)
            np.testing.assert_array_equal(net.params(), step.params())


def test_order_of_epochs_of_two_buffers():
    E, epochs, batch = 131074, 4, 65536
    log(f"training draws E={E} epochs={epochs}")
    r = np.random.default_rng(E)
    f, y = r.normal(0, 1, (E, 12)).astype(np.float32), (r.random(E) < 0.1).astype(np.float32)
    with pr.PriorNet(5) as net, pr.PriorNet(5) as step:
        net.train(f, y, epochs=epochs, batch=batch, lr=1e-3, lr_final=1e-3, pos_weight=3.0, shuffle_seed=9)
        for perm in _orders(E, epochs, 9):
            for b in range(0, E, batch):
                at = perm[b:b + batch]
                g, _ = step.gradient(f[at], y[at], 3.0)
                step.adam_step(g, 1e-3)
        np.testing.assert_array_equal(net.params(), step.params())
