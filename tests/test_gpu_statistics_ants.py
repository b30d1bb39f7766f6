"""Statistics and pheromone pass at the edges of the one-wave selection:
numbers of ants around 64, 1024 and past them, one to sixteen elites (more
elites than ants included), equal lengths in one group of 64 and across
groups, a new best-so-far and none.  Against the oracle: indices, tours,
counts and pheromone must be equal (the same fp32 operations in the same
order)."""
import numpy as np
import pytest

import oracle
import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import instances as I

from helpers import log, oracle_construct_all, oracle_problem, pack_tours, random_tau

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("better", [True, False])
@pytest.mark.parametrize("m,ras", [(1, 1), (2, 6), (5, 16), (63, 6), (64, 2), (65, 6), (130, 16), (1023, 6), (1024, 9), (1025, 6)])
def test_statistics_match_oracle(m, ras, better):
    log(f"statistics m={m} ras={ras} better={better}")
    inst = I.uniform_100(0)
    P = oracle_problem(inst)
    _, ti = oracle.pheromone_init(P, 0.5)
    some = min(m, 24)
    pm = np.array([[oracle.pm_seed(5, a, l) for l in range(64)] for a in range(some)], np.int32)
    otours, olens, _, _ = oracle_construct_all(P, ti, 0, 0, 0, 0, pm)
    r = np.random.default_rng(m)
    pick = r.integers(0, some, size=m)           # few tours: many equal lengths
    tours, lens = [otours[q] for q in pick], olens[pick]
    order = np.argsort(lens, kind="stable")
    bsf = order[-1] if better else order[0]
    packed, sizes = pack_tours(tours + [tours[bsf]], 2 * inst.n)
    bsf_len = np.float32(lens[bsf] + (1.0 if better else 0.0))
    lens = np.concatenate([lens, [bsf_len]]).astype(np.float32)
    tau0 = random_tau(inst.n, 8)
    ti0 = (tau0 * P.heur).astype(np.float32)
    with ca.GpuACO(inst, n_ants=m, seed=1, ras_ranks=ras, use_graph=False) as g:
        g.init_aco()
        it0, nrec0 = g.iteration, len(g.bsf_records())
        g.set_ants(packed, sizes, lens)
        g.set_pheromone(tau0, ti0)
        g.update_statistics()
        g.pheromone_update()
        gt, gs, gl = g.ants()
        gtau, gti = g.pheromone()
        rec, it1 = g.bsf_records(), g.iteration
    best, flag = oracle.iteration_best(lens[:m], lens[m])
    assert flag == better
    slot = best if flag else m
    all_tours = tours + [tours[bsf]]
    np.testing.assert_array_equal(gt[m, : gs[m]], all_tours[slot])
    assert gl[m] == lens[slot] and it1 == it0 + 1
    assert len(rec) == nrec0 + int(flag)
    if flag:
        assert rec[-1][0] == it0 and rec[-1][1] == lens[best]
    # elites: the best-so-far slot, then ants by length, ties to the lowest
    # index, ant 0 when the ants run out
    el = [m] + [int(a) for a in np.argsort(lens[:m], kind="stable")[: ras - 1]]
    el += [0] * (ras - len(el))
    after = lens.copy()
    after[m] = lens[slot]
    etours = [all_tours[slot] if e == m else all_tours[e] for e in el]
    otau, oti = oracle.pheromone_update(P, tau0, etours, [after[e] for e in el])
    np.testing.assert_array_equal(gtau, otau)
    np.testing.assert_array_equal(gti, oti)
