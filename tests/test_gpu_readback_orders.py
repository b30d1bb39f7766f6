"""Transfers of very different sizes through one context's pinned buffers, in
several orders (a buffer's size follows the context's, and the second one is
made by the first transfer that fills the first): everything read must equal
what a context reads that does nothing else, and what is written must come
back.  Bytes only: equal."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import instances as I

from helpers import log

pytestmark = pytest.mark.gpu


def _context(inst, ants):
    g = ca.GpuACO(inst, n_ants=ants, k=6, seed=4, selection=ca.SEL_KNN, rng=ca.RNG_PHILOX, ls_flags=0, use_graph=False)
    g.init_aco()
    g.run(2)
    return g


def _ants(g):
    tours, sizes, lens = g.ants()
    tours[np.arange(tours.shape[1])[None, :] >= sizes[:, None]] = 0
    return [tours, sizes, lens]


CALLS = {"best": lambda g: list(g.best()), "ants": _ants, "trail": lambda g: list(g.pheromone()),
         "setup": lambda g: list(g.setup_arrays().values())}


def _same(a, b, what):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y, err_msg=what)


# matrices of 3 KB, 90 KB, 510 to 530 KB (n = 361 .. 368) and 4 MB; tours of 2 KB to 1 MB
@pytest.mark.parametrize("n,ants", [(26, 9), (26, 400), (150, 3), (361, 64), (366, 180), (1001, 130)])
def test_transfers_in_any_order(n, ants):
    log(f"transfers n={n} ants={ants}")
    inst = I.mixed_1000(2).subset(n)
    want = {}
    for what, call in CALLS.items():
        with _context(inst, ants) as g:
            want[what] = call(g)
    for order in (("best", "ants", "trail", "setup", "best", "ants"), ("setup", "trail", "best", "ants"),
                  ("ants", "best", "setup", "trail", "setup")):
        with _context(inst, ants) as g:
            for what in order:
                _same(CALLS[what](g), want[what], f"{what} in {order}")
            # other matrices, whatever was read before
            tau, ti = want["trail"]
            g.set_pheromone(ti.T.copy(), tau.T.copy())
            _same(CALLS["trail"](g), [ti.T, tau.T], "trail after set_pheromone")
            _same(CALLS["best"](g), want["best"], "best after set_pheromone")
    with _context(inst, ants) as g:   # written before anything is read
        g.set_pheromone(ti.T.copy(), tau.T.copy())
        _same(CALLS["trail"](g), [ti.T, tau.T], "trail after set_pheromone alone")
