"""I-Roulette construction with several waves per ant where the roulette has
no mass at the depot and the ant's waves pick the next node together
(largest total_info, ties to the lowest index): no mass anywhere, and mass in
one entry of fifty.  Rows in LDS and in global memory, four and eight waves,
one to eight nodes per lane, with and without a route-length limit.  Against
the oracle; the same draws, comparisons and additions in the same order, so
everything must be equal."""
import math

import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_construct_all, oracle_problem

pytestmark = pytest.mark.gpu

ANTS = 4


@pytest.mark.parametrize("limited", [False, True])
@pytest.mark.parametrize("mass", ["none", "few"])
@pytest.mark.parametrize("n", [50, 130, 136, 200, 300, 700, 1100, 2100])
def test_picks_without_mass_match_oracle(n, mass, limited):
    log(f"I-Roulette fallback n={n} mass={mass} limited={limited}")
    r = np.random.default_rng(n)
    xy = r.integers(0, 200, size=(n, 2)).astype(np.float64) * 4.0
    dem = np.concatenate([[0], r.integers(1, 30, size=n - 1)]).astype(np.int32)
    lim, svc = math.inf, 0.0
    if limited:
        svc = 3.0
        lim = math.ceil(2.4 * float(np.hypot(*(xy - xy[0]).T).max()) + 4 * svc)
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 150, ca.DIST_NINT, max_dist=lim, service_time=svc)
    P = oracle_problem(inst)
    ti = np.zeros((n, n), np.float32)
    if mass == "few":
        # few distinct values, so that picks between equal ones occur too;
        # none in half of the depot's row
        ti = np.where(r.random((n, n)) < 0.02, r.integers(1, 4, size=(n, n)), 0).astype(np.float32)
        ti[0, n // 2:] = 0.0
    with ca.GpuACO(inst, n_ants=ANTS, k=0, seed=3, ls_flags=0, use_graph=False, tau0_rule=ca.TAU0_NN_TOUR) as g:
        g.init_aco()
        g.set_pheromone(np.full((n, n), 0.5, np.float32), ti)
        pm = g.rng_state()
        g.construct_solutions()
        tours, sizes, lens = g.ants()
        after = g.rng_state()
        g.update_statistics()
        fallbacks = g.counters()["fallbacks"]
    otours, olens, opm, ofb = oracle_construct_all(P, ti, 0, 0, 3, 0, pm)
    assert ofb >= ANTS * (n - 1 if mass == "none" else 1)
    np.testing.assert_array_equal(after, opm)
    for a, t in enumerate(otours):
        assert sizes[a] == len(t), a
        np.testing.assert_array_equal(tours[a, : sizes[a]], t, err_msg=f"ant {a}")
        assert lens[a] == olens[a]
    assert fallbacks == ofb
