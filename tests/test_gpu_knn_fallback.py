"""Candidate roulette whose fallback keeps the nodes in registers, against
the oracle: sizes on both sides of 8 and 16 nodes per lane and of whole
rounds of 64, narrow candidate rows (most steps fall back), equal
total_info values, with and without a route-length limit, few and many ants
(every load issued, or only those of chunks with something feasible), rows
from global memory and from LDS.  Whole numbers and the same additions in
the same order: everything must be equal."""
import math

import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_construct_all, oracle_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ants,limited,apb", [
    (4, 4, False, 0), (64, 8, True, 0), (65, 8, False, 4), (65, 1032, False, 0), (129, 1028, True, 0),
    (511, 8, True, 0), (512, 8, False, 2), (513, 8, True, 0), (513, 8, False, 4), (1024, 4, False, 0),
    (1024, 4, True, 0), (1025, 4, False, 0), (1025, 4, True, 0), (700, 1028, False, 0)])
@pytest.mark.parametrize("rng", [ca.RNG_PHILOX, ca.RNG_PARK_MILLER])
def test_fallback_matches_oracle(n, ants, limited, apb, rng):
    log(f"fallback n={n} ants={ants} limited={limited} apb={apb} rng={rng}")
    r = np.random.default_rng(n + ants)
    xy = r.integers(0, 25, size=(n, 2)).astype(np.float64) * 30.0   # few places: equal values
    dem = np.concatenate([[0], r.integers(1, 30, size=n - 1)]).astype(np.int32)
    lim, svc = math.inf, 0.0
    if limited:
        svc = 2.0
        lim = math.ceil(2.5 * float(np.hypot(*(xy - xy[0]).T).max()) + 4 * svc)
    k = 2
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 120, ca.DIST_NINT, max_dist=lim, service_time=svc)
    P = oracle_problem(inst, k=k)
    _, ti = oracle.pheromone_init(P, 0.5)
    with ca.GpuACO(inst, n_ants=ants, k=k, seed=3, selection=ca.SEL_KNN, rng=rng, ls_flags=0, use_graph=False,
                   tau0_rule=ca.TAU0_NN_TOUR) as g:
        g.init_aco()
        g.pheromone_init(0.5)
        if apb:
            g.set_launch_shape(4, 16, 0, apb, 0)
        pm = g.rng_state()
        g.construct_solutions()
        tours, sizes, lens = g.ants()
        g.update_statistics()
        fallbacks = g.counters()["fallbacks"]
    few = min(ants, 24)   # the oracle's share of many ants
    otours, olens, _, ofb = oracle_construct_all(P, ti, 1, int(rng == ca.RNG_PHILOX), 3, 0, pm[:few])
    for a, t in enumerate(otours):
        assert sizes[a] == len(t), a
        np.testing.assert_array_equal(tours[a, : sizes[a]], t, err_msg=f"ant {a}")
        assert lens[a] == olens[a]
    assert ofb > 0 or n < 10
    if few == ants:
        assert fallbacks == ofb
    else:
        for a in range(few, ants, 97):
            assert inst.check_solution(tours[a, : sizes[a]])
