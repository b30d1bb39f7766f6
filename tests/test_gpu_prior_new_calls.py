"""The prior's calls through its pinned memory as it grows: on one network,
calls that fit the smallest part, one part of 512 KB and two of them, in
rising and falling order and mixed (gradient, training, dense multiplier),
equal, bit for bit, the same calls on networks of their own."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import instances as I
from cvrp_aco_ocl_amd import prior as pr

from helpers import log

pytestmark = pytest.mark.gpu

# rows of a part of 32 KB and of one of 512 KB, and their neighbours
SIZES = [1, 630, 631, 10082, 10083, 30000]


def _gradient(net, E):
    r = np.random.default_rng(E)
    g, loss = net.gradient(r.normal(0, 1, (E, 12)), r.random(E) < 0.1, 3.0)
    return [g, loss]


def _train(net, E):
    start = net.params()
    r = np.random.default_rng(E)
    losses = net.train(r.normal(0, 1, (E, 12)), r.random(E) < 0.1, epochs=2, batch=4096, shuffle_seed=7)
    out = [net.params(), losses]
    net.set_params(start)   # the moments too
    return out


def _build(net, n):
    inst = I.mixed_1000(1).subset(n)
    k = min(8, n - 2)
    return [net.build(inst, inst.nn_lists(k), k)]


CALLS = [(_gradient, E) for E in SIZES] + [(_train, E) for E in SIZES] + [(_build, n) for n in (10, 90, 91, 362, 363, 600)]


@pytest.mark.parametrize("order", ["rising", "falling", "mixed"])
def test_growing_calls(order):
    log(f"prior calls {order}")
    calls = list(CALLS)
    if order == "rising":
        calls.sort(key=lambda c: c[1])
    elif order == "falling":
        calls.sort(key=lambda c: -c[1])
    else:
        calls = [calls[i] for i in np.random.default_rng(3).permutation(len(calls))]
    with pr.PriorNet(5) as net:
        for call, size in calls:
            got = call(net, size)
            with pr.PriorNet(5) as own:
                want = call(own, size)
            for x, y in zip(got, want):
                np.testing.assert_array_equal(x, y, err_msg=f"{call.__name__} {size}")
