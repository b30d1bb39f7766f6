"""Instances with one distance past the 16-bit relocate's range, or one node
at a distance from itself, wherever in its row it stands (the check takes
eight entries at a time and the rest one by one): the search must be exact,
against the oracle.  Whole numbers: equal."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_problem, pack_tours

pytestmark = pytest.mark.gpu

ANTS, ROUTES = 3, 30


@pytest.mark.parametrize("where", ["last", "first", "eighth", "diagonal"])
@pytest.mark.parametrize("n", [488, 489, 492, 495])
def test_one_entry_out_of_range(n, where):
    log(f"packed range n={n} where={where}")
    r = np.random.default_rng(n)
    d = np.triu(r.integers(7000, 8191, size=(n, n)), 1)
    d = d + d.T
    if where == "diagonal":
        d[n - 1, n - 1] = 5
    else:
        a, b = {"last": (n - 2, n - 1), "first": (1, 2), "eighth": (8, 15)}[where]
        d[a, b] = d[b, a] = 60000
    d = d.astype(np.float32)
    dem = np.concatenate([[0], r.integers(1, 31, size=n - 1)]).astype(np.int32)
    tours = []
    for _ in range(ANTS):
        parts = np.array_split(r.permutation(np.arange(1, n)), ROUTES)
        tours.append(np.concatenate([np.concatenate([[0], p]) for p in parts] + [[0]]).astype(np.int32))
    inst = Instance(n=n, x=np.zeros(n), y=np.zeros(n), demand=dem, capacity=500, dist=d)
    P = oracle_problem(inst)
    lens = np.array([d[t[:-1], t[1:]].sum() for t in tours + tours[:1]], np.float32)
    packed, sizes = pack_tours(tours + [tours[0]], 2 * n)
    with ca.GpuACO(inst, n_ants=ANTS, seed=1, ls_flags=ca.LS_RELOCATE, use_graph=False) as g:
        g.init_aco()
        g.set_launch_shape(4, 16, 0, 0, 1)
        g.set_ants(packed, sizes, lens)
        g.local_search()
        got, gsizes, glens = g.ants()
    for a in range(ANTS):
        t, L, _ = P.local_search(tours[a], ca.LS_RELOCATE)
        assert gsizes[a] == len(t), a
        np.testing.assert_array_equal(got[a, : len(t)], t, err_msg=f"ant {a}")
        assert glens[a] == np.float32(L), (a, glens[a], L)
