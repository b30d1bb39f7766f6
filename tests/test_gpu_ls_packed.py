"""Local search at the edges of its 16-bit relocate, against the oracle:
distance matrices at and past the largest distance and demand that take it,
a non-zero diagonal (which does not), tours around one and two lanes' worth
of positions, around one trip (512 edges) and past a block's reach in one
shift (4 positions per thread), one route and many, with and without a
route-length limit.  Whole numbers: tours and evaluated-move counts must be
equal, and so must the lengths (sums in the same order)."""
import math

import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_construct_all, oracle_problem, pack_tours

pytestmark = pytest.mark.gpu

ANTS = 12
RELOCATE, ALL = ca.LS_RELOCATE, ca.LS_2OPT | ca.LS_SWAP | ca.LS_RELOCATE

# n, largest distance, largest demand, diagonal, routes, limited, waves, flags
CASES = [
    (4, 8190, 9, 0, 1, False, 4, RELOCATE),
    (8, 8190, 8191, 0, 2, False, 4, ALL),
    (9, 8191, 9, 0, 2, False, 4, ALL),          # longest distance: general path
    (15, 8190, 8192, 0, 3, False, 8, ALL),      # largest demand: general path
    (17, 8190, 8191, 0, 3, True, 16, RELOCATE),
    (33, 300, 9, 7, 4, False, 4, ALL),          # diagonal: general path
    (64, 8190, 40000, 0, 2, False, 8, ALL),     # demands and loads past 16 bits: general path
    (64, 8190, 8191, 0, 1, True, 8, ALL),       # a load past 16 bits
    (130, 100, 5, 0, 100, False, 12, ALL),
    (509, 8190, 30, 0, 2, False, 4, RELOCATE),
    (512, 8190, 30, 0, 1, True, 8, RELOCATE),
    (700, 40, 30, 0, 350, False, 4, RELOCATE),  # tour past 4 positions per thread
    (1100, 2000, 30, 0, 60, True, 4, RELOCATE),
]


@pytest.mark.parametrize("n,far,big,diag,routes,limited,waves,flags", CASES)
def test_local_search_edges_match_oracle(n, far, big, diag, routes, limited, waves, flags):
    log(f"packed relocate n={n} far={far} big={big} diag={diag} routes={routes} limited={limited} waves={waves}")
    r = np.random.default_rng(n + far)
    d = np.triu(r.integers(0, far + 1, size=(n, n)), 1)
    d[0, n - 1] = far
    d = d + d.T + diag * np.eye(n, dtype=d.dtype)
    dem = np.concatenate([[0], r.integers(1, big + 1, size=n - 1)]).astype(np.int32)
    dem[1] = big
    cap = max(math.ceil(int(dem.sum()) / routes) + (big if routes > 1 else 0), big)
    svc = 3.0 if limited else 0.0
    lim = 2.0 * far + svc + far * (n // (2 * routes)) * 0.4 if limited else math.inf
    inst = Instance(n=n, x=np.zeros(n), y=np.zeros(n), demand=dem, capacity=cap, dist=d.astype(np.float32),
                    max_dist=lim, service_time=svc)
    P = oracle_problem(inst)
    _, ti = oracle.pheromone_init(P, 0.5)
    pm = np.array([[oracle.pm_seed(n, a, l) for l in range(64)] for a in range(ANTS)], np.int32)
    otours, olens, _, _ = oracle_construct_all(P, ti, 0, 0, 0, 0, pm)
    packed, sizes = pack_tours(otours + [otours[0]], 2 * n)
    with ca.GpuACO(inst, n_ants=ANTS, seed=1, ls_flags=flags, use_graph=False) as g:
        g.init_aco()
        g.set_launch_shape(waves, 16 if waves < 16 else 32, 0, 0, 1)
        g.set_ants(packed, sizes, np.concatenate([olens, olens[:1]]).astype(np.float32))
        g.local_search()
        tours, gsizes, glens = g.ants()
        g.update_statistics()   # folds the per-ant counters into the totals
        evals = g.counters()["ls_evals"]
    total = 0
    for a in range(ANTS):
        t, L, ev = P.local_search(otours[a], flags)
        total += ev
        assert gsizes[a] == len(t), a
        np.testing.assert_array_equal(tours[a, : len(t)], t, err_msg=f"ant {a}")
        assert glens[a] == np.float32(L), (a, glens[a], L)
    assert evals == total
