"""I-Roulette construction with several waves per ant, against the oracle:
instance sizes on both sides of each choice of waves and nodes per lane, and
around the largest instances whose matrices are held in LDS, with and
without a route-length limit.  The same draws and the same additions in the
same order: tours, lengths, lane states and fallbacks must be equal."""
import math

import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_construct_all, oracle_problem

pytestmark = pytest.mark.gpu

ANTS = 6


@pytest.mark.parametrize("limited", [False, True])
@pytest.mark.parametrize("n", [3, 5, 63, 64, 65, 128, 129, 136, 144, 192, 200, 256, 257, 512, 513, 1024, 1025, 2049])
def test_iroulette_matches_oracle(n, limited):
    log(f"I-Roulette n={n} limited={limited}")
    r = np.random.default_rng(n)
    # a few grid points: equal distances, so equal probabilities' ties too
    xy = r.integers(0, 40, size=(n, 2)).astype(np.float64) * 20.0
    dem = np.concatenate([[0], r.integers(1, 30, size=n - 1)]).astype(np.int32)
    lim, svc = math.inf, 0.0
    if limited:
        far = float(np.hypot(*(xy - xy[0]).T).max())
        svc = 3.0
        lim = math.ceil(2.4 * far + 4 * svc)
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 150, ca.DIST_NINT, max_dist=lim, service_time=svc)
    P = oracle_problem(inst)
    _, ti = oracle.pheromone_init(P, 0.5)
    with ca.GpuACO(inst, n_ants=ANTS, k=0, seed=3, ls_flags=0, use_graph=False, tau0_rule=ca.TAU0_NN_TOUR) as g:
        g.init_aco()
        g.pheromone_init(0.5)
        pm = g.rng_state()
        g.construct_solutions()
        tours, sizes, lens = g.ants()
        after = g.rng_state()
        g.update_statistics()
        fallbacks = g.counters()["fallbacks"]
    otours, olens, opm, ofb = oracle_construct_all(P, ti, 0, 0, 3, 0, pm)
    np.testing.assert_array_equal(after, opm)
    for a, t in enumerate(otours):
        assert sizes[a] == len(t), a
        np.testing.assert_array_equal(tours[a, : sizes[a]], t, err_msg=f"ant {a}")
        assert lens[a] == olens[a]
    assert fallbacks == ofb
