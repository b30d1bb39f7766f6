"""Candidate roulette with a route-length limit and more ants than the device
has SIMDs (the full-row pick reads only chunks of nodes with something
feasible), at the sizes whose pick keeps sixteen nodes per lane: the smallest
and the largest of them and both sides of whole rounds of 64.  The first and
the last ants against the oracle, every tour checked; everything must be
equal."""
import math

import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_construct_all, oracle_problem

pytestmark = pytest.mark.gpu

ANTS, SOME = 1100, 10


@pytest.mark.parametrize("rng", [ca.RNG_PHILOX, ca.RNG_PARK_MILLER])
@pytest.mark.parametrize("n", [513, 640, 641, 1023, 1024])
def test_limited_pick_of_many_ants(n, rng):
    log(f"narrow limited pick n={n} rng={rng}")
    r = np.random.default_rng(n)
    xy = r.integers(0, 25, size=(n, 2)).astype(np.float64) * 30.0   # few places: equal values
    dem = np.concatenate([[0], r.integers(1, 30, size=n - 1)]).astype(np.int32)
    svc = 2.0
    lim = math.ceil(2.5 * float(np.hypot(*(xy - xy[0]).T).max()) + 4 * svc)
    k = 3
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 120, ca.DIST_NINT, max_dist=lim, service_time=svc)
    P = oracle_problem(inst, k=k)
    _, ti = oracle.pheromone_init(P, 0.5)
    with ca.GpuACO(inst, n_ants=ANTS, k=k, seed=3, selection=ca.SEL_KNN, rng=rng, ls_flags=0, use_graph=False,
                   tau0_rule=ca.TAU0_NN_TOUR) as g:
        g.init_aco()
        g.pheromone_init(0.5)
        pm = g.rng_state()
        g.construct_solutions()
        tours, sizes, lens = g.ants()
    tiknn = oracle.gather_knn(P, ti)
    picks = 0
    for a in list(range(SOME)) + list(range(ANTS - SOME, ANTS)):
        t, L, fb = P.construct_ant(ti, tiknn, 1, int(rng == ca.RNG_PHILOX), 3, 0, a, pm[a].copy())
        assert sizes[a] == len(t), a
        np.testing.assert_array_equal(tours[a, : sizes[a]], t, err_msg=f"ant {a}")
        assert lens[a] == L
        picks += fb
    assert picks > 0
    for a in range(ANTS):
        assert inst.check_solution(tours[a, : sizes[a]]), a
