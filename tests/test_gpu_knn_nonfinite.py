"""Candidate roulette over total_info that does not add up to a positive
number: infinities (trails of a colony whose tours have length 0), NaN and
negative values (set from outside).  A candidate's value counts 1 or 0 times
as it is feasible or not, so an infinity that is not feasible makes the total
NaN; a total that is not above 0, NaN included, is no wheel, and the step
takes the full-row pick (largest bits, ties to the lowest index).  An
infinite total picks the last feasible candidate whatever is drawn.

Negative and overflowing values against the oracle; where every row has an
infinite or NaN candidate, no draw matters and the tours follow from the
rule above, written out here.  Rows from global memory and from LDS, the pick
from registers and past them, with and without a route-length limit.  Whole
numbers and the same additions in the same order: everything must be equal."""
import math

import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_construct_all, oracle_problem

pytestmark = pytest.mark.gpu

ANTS, K = 8, 8


def tour_without_draws(inst, ti, nn):
    """Tour and number of full-row picks where every row of ti has a
    candidate that is infinite or NaN."""
    n, f32 = inst.n, np.float32
    bits = np.ascontiguousarray(ti).view(np.uint32)
    seen = np.zeros(n, bool)
    seen[0] = True
    tour, cur, load, rdist, picks = [0], 0, 0, f32(0), 0
    while not seen.all():
        to = (f32(rdist) + (inst.dist[cur] + f32(inst.service_time))).astype(f32) + inst.dist[:, 0]
        ok = ~seen & (load + inst.demand <= inst.capacity) & (to <= f32(inst.max_dist))
        c = nn[cur, :K]
        bad = np.isnan(ti[cur, c]) | (np.isinf(ti[cur, c]) & ~ok[c])
        if bad.any() or not ok[c].any():
            # one more than the bits, in 32 bits: all ones come last
            w = int(np.argmax(np.where(ok, (bits[cur].astype(np.int64) + 1) & 0xFFFFFFFF, -1))) if ok.any() else 0
            picks += 1
        else:
            w = int(c[ok[c] & (ti[cur, c] > 0)][-1])
        if w == 0:
            load, rdist = 0, f32(0)
        else:
            load, rdist = load + int(inst.demand[w]), f32(rdist + (inst.dist[cur, w] + f32(inst.service_time)))
        seen[w] = True
        tour.append(w)
        cur = w
    return tour + [0], picks


@pytest.mark.parametrize("kind", ["inf", "nan", "negative", "overflow"])
@pytest.mark.parametrize("rng", [ca.RNG_PHILOX, ca.RNG_PARK_MILLER])
@pytest.mark.parametrize("n,limited,apb", [(40, False, 0), (40, True, 0), (70, False, 2), (70, False, 4), (600, False, 0),
                                           (600, True, 0), (600, False, 4), (1100, False, 0), (1100, False, 1)])
def test_wheel_without_a_positive_total(n, limited, apb, rng, kind):
    log(f"total_info {kind} n={n} limited={limited} apb={apb} rng={rng}")
    r = np.random.default_rng(n)
    xy = r.integers(0, 300, size=(n, 2)).astype(np.float64)
    dem = np.concatenate([[0], r.integers(1, 30, size=n - 1)]).astype(np.int32)
    lim, svc = math.inf, 0.0
    if limited:
        svc = 2.0
        lim = math.ceil(2.5 * float(np.hypot(*(xy - xy[0]).T).max()) + 4 * svc)
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 150, ca.DIST_NINT, max_dist=lim, service_time=svc)
    P = oracle_problem(inst, k=K)
    nn = inst.nn_lists(K)
    ti = r.uniform(0.1, 1.0, size=(n, n)).astype(np.float32)
    if kind == "overflow":
        ti *= np.float32(3e38)
    elif kind == "negative":
        ti[r.random((n, n)) < 0.2] = -4.0
    else:
        ti[r.random((n, n)) < 0.05] = np.inf
        at = nn[np.arange(n), r.integers(0, K, size=n)]
        # the depot's first candidates too, so that both ways of a step occur
        ti[np.arange(n), at] = np.where(np.arange(n) % 2 == 0, np.inf, np.nan) if kind == "nan" else np.inf
    with ca.GpuACO(inst, n_ants=ANTS, k=K, seed=3, selection=ca.SEL_KNN, rng=rng, ls_flags=0, use_graph=False,
                   tau0_rule=ca.TAU0_NN_TOUR) as g:
        g.init_aco()
        if apb:
            g.set_launch_shape(4, 16, 0, apb, 0)
        g.set_pheromone(np.full((n, n), 0.5, np.float32), ti)
        pm = g.rng_state()
        g.construct_solutions()
        tours, sizes, lens = g.ants()
        after = g.rng_state()
        g.update_statistics()
        fallbacks = g.counters()["fallbacks"]
    if kind in ("negative", "overflow"):
        want, olens, opm, picks = oracle_construct_all(P, ti, 1, int(rng == ca.RNG_PHILOX), 3, 0, pm)
        if rng == ca.RNG_PARK_MILLER:
            np.testing.assert_array_equal(after, opm)
        np.testing.assert_array_equal(lens[:ANTS], olens)
    else:
        t, picks = tour_without_draws(inst, ti, nn)
        want, picks = [t] * ANTS, ANTS * picks
    for a, t in enumerate(want):
        assert sizes[a] == len(t), a
        np.testing.assert_array_equal(tours[a, : sizes[a]], t, err_msg=f"ant {a}")
    assert fallbacks == picks > 0


@pytest.mark.parametrize("part", [1.0, 0.6])
@pytest.mark.parametrize("n,limited,apb", [(40, False, 0), (40, True, 0), (70, False, 4), (600, False, 0), (600, True, 0),
                                           (600, False, 2), (1024, True, 0), (1100, False, 0)])
def test_bits_all_ones(n, limited, apb, part):
    """NaN with every bit set, everywhere or in most entries, the rest 0 (at
    every candidate, so no draw matters): the last of all values, but a node
    that has it is still placed."""
    log(f"total_info all ones n={n} limited={limited} apb={apb} part={part}")
    r = np.random.default_rng(n)
    xy = r.integers(0, 300, size=(n, 2)).astype(np.float64)
    dem = np.concatenate([[0], r.integers(1, 30, size=n - 1)]).astype(np.int32)
    lim, svc = math.inf, 0.0
    if limited:
        svc = 2.0
        lim = math.ceil(2.5 * float(np.hypot(*(xy - xy[0]).T).max()) + 4 * svc)
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 150, ca.DIST_NINT, max_dist=lim, service_time=svc)
    nn = inst.nn_lists(K)
    bits = np.where(r.random((n, n)) < part, 0xFFFFFFFF, 0).astype(np.uint32)
    bits[np.arange(n)[:, None], nn] = 0xFFFFFFFF
    ti = bits.view(np.float32)
    with ca.GpuACO(inst, n_ants=ANTS, k=K, seed=3, selection=ca.SEL_KNN, rng=ca.RNG_PHILOX, ls_flags=0, use_graph=False,
                   tau0_rule=ca.TAU0_NN_TOUR) as g:
        g.init_aco()
        if apb:
            g.set_launch_shape(4, 16, 0, apb, 0)
        g.set_pheromone(np.full((n, n), 0.5, np.float32), ti)
        g.construct_solutions()
        tours, sizes, _ = g.ants()
    t, _ = tour_without_draws(inst, ti, nn)
    for a in range(ANTS):
        assert sizes[a] == len(t), a
        np.testing.assert_array_equal(tours[a, : sizes[a]], t, err_msg=f"ant {a}")


def test_customers_in_one_place():
    """Every distance 0: tours of length 0, so every trail is infinite."""
    n = 60
    log("one place")
    dem = np.concatenate([[0], np.arange(1, n) % 29 + 1]).astype(np.int32)
    inst = Instance.from_coords(np.full(n, 5.0), np.full(n, 5.0), dem, 150, ca.DIST_NINT)
    with ca.GpuACO(inst, n_ants=ANTS, k=K, seed=3, selection=ca.SEL_KNN, rng=ca.RNG_PHILOX, ls_flags=0,
                   use_graph=False, tau0_rule=ca.TAU0_FIRST_COLONY) as g:
        g.init_aco()
        _, ti = g.pheromone()
        assert np.isinf(ti).all()
        g.construct_solutions()
        tours, sizes, lens = g.ants()
    t, _ = tour_without_draws(inst, ti, inst.nn_lists(K))
    for a in range(ANTS):
        assert sizes[a] == len(t) and lens[a] == 0.0, a
        np.testing.assert_array_equal(tours[a, : sizes[a]], t, err_msg=f"ant {a}")
