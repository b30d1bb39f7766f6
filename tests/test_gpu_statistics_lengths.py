"""Elites where ant lengths are not positive numbers (aco_set_ants takes any):
lengths are compared by their bits, so infinity comes behind every positive
one and before negative ones and NaN, and a smallest value of infinity, which
a taken ant counts as too, makes ant 0 the elite.  One wave's selection (up
to 1024 ants) and the block's (more).  The same fp32 operations in the same
order as the oracle's: equal."""
import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import instances as I

from helpers import log, oracle_construct_all, oracle_problem, pack_tours, random_tau

pytestmark = pytest.mark.gpu

RAS = 5


def _elites(lens, m):
    bits = lens[:m].view(np.uint32).astype(np.uint64).copy()
    out = [m]
    for _ in range(1, RAS):
        a = int(np.argmin(bits))
        a = 0 if bits[a] == 0x7F800000 else a
        out.append(a)
        bits[a] = 0x7F800000
    return out


@pytest.mark.parametrize("kind", ["negative", "infinite", "mixed"])
@pytest.mark.parametrize("m", [7, 70, 1024, 1100])
def test_elites_of_any_lengths(m, kind):
    log(f"statistics lengths m={m} kind={kind}")
    inst = I.uniform_100(0)
    P = oracle_problem(inst)
    _, ti = oracle.pheromone_init(P, 0.5)
    pm = np.array([[oracle.pm_seed(5, a, l) for l in range(64)] for a in range(7)], np.int32)
    base, _, _, _ = oracle_construct_all(P, ti, 0, 0, 0, 0, pm)
    r = np.random.default_rng(m)
    tours = [base[a % 7] for a in range(m)] + [base[0]]
    lens = np.empty(m + 1, np.float32)
    lens[:m] = -r.permutation(np.arange(100, 100 + m))
    if kind == "infinite":
        lens[:m] = np.inf
        lens[m // 2] = 3000.0
    elif kind == "mixed":
        lens[1:m:3] = np.inf
        lens[2] = 2500.0
    lens[m] = 2000.0
    packed, sizes = pack_tours(tours, 2 * inst.n)
    tau0 = random_tau(inst.n, 8)
    with ca.GpuACO(inst, n_ants=m, seed=1, ras_ranks=RAS, use_graph=False) as g:
        g.init_aco()
        g.set_ants(packed, sizes, lens)
        g.set_pheromone(tau0, (tau0 * P.heur).astype(np.float32))
        g.update_statistics()
        g.pheromone_update()
        gt, gs, gl = g.ants()
        gtau, _ = g.pheromone()
    best = int(np.argmin(lens[:m].view(np.uint32)))
    flag = lens[best] - lens[m] < -0.001
    after = lens.copy()
    etours = list(tours)
    if flag:
        after[m], etours[m] = lens[best], tours[best]
    assert gl[m] == after[m]
    np.testing.assert_array_equal(gt[m, : gs[m]], etours[m])
    el = _elites(lens, m)
    otau, _ = oracle.pheromone_update(P, tau0, [etours[e] for e in el], [after[e] for e in el])
    np.testing.assert_array_equal(gtau, otau)
