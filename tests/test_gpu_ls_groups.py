"""2-opt with 8, 4, 2 or 1 positions at a time, against the oracle: numbers
of routes on both sides of each choice for blocks of 4, 8 and 16 waves, and
routes around and past the 64 scan indices a group looks at at once.  Whole
numbers: tours, lengths and evaluated-move counts must be equal."""
import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_problem, pack_tours

pytestmark = pytest.mark.gpu

ANTS = 8


@pytest.mark.parametrize("nint", [True, False])
@pytest.mark.parametrize("waves,routes,length", [
    (4, 1, 63), (4, 1, 64), (4, 2, 65), (4, 4, 40), (4, 5, 40), (4, 8, 20), (4, 9, 20), (4, 16, 7),
    (4, 17, 7), (4, 4, 130), (8, 8, 12), (8, 9, 12), (8, 16, 33), (8, 17, 33), (8, 32, 3), (8, 33, 3),
    (16, 16, 9), (16, 17, 40), (16, 40, 1)])
def test_2opt_matches_oracle(waves, routes, length, nint):
    log(f"2-opt waves={waves} routes={routes} length={length} nint={nint}")
    n = routes * length + 1
    r = np.random.default_rng(100 * routes + length)
    xy = r.integers(0, 1001, size=(n, 2)).astype(np.float64)
    dem = np.ones(n, np.int32)
    dem[0] = 0
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, length, ca.DIST_NINT if nint else ca.DIST_FLOAT)
    P = oracle_problem(inst)
    tours = []
    for _ in range(ANTS + 1):
        c = r.permutation(np.arange(1, n)).reshape(routes, length)
        tours.append(np.concatenate([np.pad(c, ((0, 0), (1, 0))).ravel(), [0]]).astype(np.int32))
    packed, sizes = pack_tours(tours, 2 * n)
    lens = np.array([inst.dist[t[:-1], t[1:]].sum() for t in tours], np.float32)
    with ca.GpuACO(inst, n_ants=ANTS, seed=1, ls_flags=ca.LS_2OPT, use_graph=False) as g:
        g.init_aco()
        g.set_launch_shape(waves, 16 if waves < 16 else 32, 0, 0, int(nint))
        g.set_ants(packed, sizes, lens)
        g.local_search()
        got, gsizes, glens = g.ants()
        g.update_statistics()   # folds the per-ant counters into the totals
        evals = g.counters()["ls_evals"]
    total = 0
    for a in range(ANTS):
        t, L, ev = P.local_search(tours[a], ca.LS_2OPT)
        total += ev
        assert gsizes[a] == len(t), a
        np.testing.assert_array_equal(got[a, : len(t)], t, err_msg=f"ant {a}")
        assert glens[a] == np.float32(L), (a, glens[a], L)
    assert evals == total
