"""Which tours the 16-bit relocate takes, for every number of waves, with and
without a route-length limit, by itself and behind a swap: tours one position
short of the line, on it and past it, and past it tours at the edges of a
trip (512 edges), of a lane's eight positions and of a block's reach in one
shift (4 positions per thread).  Against the oracle.  Whole numbers: tours
and evaluated-move counts must be equal, and so must the lengths (sums in the
same order)."""
import math

import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd.solver import Instance

from helpers import log, oracle_problem, pack_tours

pytestmark = pytest.mark.gpu

ANTS = 4
ALONE, FULL = ca.LS_RELOCATE, ca.LS_2OPT | ca.LS_SWAP | ca.LS_RELOCATE
LINE = {(4, False, FULL): 300, (4, True, FULL): 360, (8, False, FULL): 480, (8, True, FULL): 560, (12, False, FULL): 780,
        (12, True, FULL): 720, (16, False, FULL): 830, (16, True, FULL): 830, (4, False, ALONE): 400,
        (4, True, ALONE): 480, (8, False, ALONE): 768, (8, True, ALONE): 650, (12, False, ALONE): 832,
        (12, True, ALONE): 900, (16, False, ALONE): 850, (16, True, ALONE): 1024}
CASES = [(w, lim, at + d, fl) for (w, lim, fl), at in LINE.items() for d in (-1, 0, 1)]
PAST = [(4, False, s) for s in (511, 512, 513, 514, 1023, 1025, 1030, 1537)] + [(4, True, s) for s in (513, 520, 1025)]
PAST += [(8, False, s) for s in (1023, 1024, 1025)] + [(12, True, s) for s in (1025, 1029)] + [(16, False, 1031)]
CASES += [(*c, fl) for c in PAST for fl in (ALONE, FULL)]


@pytest.mark.parametrize("waves,limited,positions,flags", CASES)
def test_relocate_at_the_line(waves, limited, positions, flags):
    log(f"relocate waves={waves} limited={limited} positions={positions} flags={flags}")
    r = np.random.default_rng(positions + waves)
    routes = positions // 13
    n = positions - routes
    d = np.triu(r.integers(1, 8191, size=(n, n)), 1)
    d = (d + d.T).astype(np.float32)
    dem = np.concatenate([[0], r.integers(1, 31, size=n - 1)]).astype(np.int32)
    tours = []
    for _ in range(ANTS):
        parts = np.array_split(r.permutation(np.arange(1, n)), routes)
        tours.append(np.concatenate([np.concatenate([[0], p]) for p in parts] + [[0]]).astype(np.int32))
        assert len(tours[-1]) == positions
    loads = [dem[part].sum() for t in tours for part in np.split(t, np.flatnonzero(t == 0)[1:-1])]
    svc, lim = 0.0, math.inf
    if limited:
        svc = 3.0
        ends = [np.flatnonzero(t == 0) for t in tours]
        lim = float(max(d[t[a:b], t[a + 1:b + 1]].sum() + svc * (b - a - 1)
                        for t, z in zip(tours, ends) for a, b in zip(z[:-1], z[1:])))
    inst = Instance(n=n, x=np.zeros(n), y=np.zeros(n), demand=dem, capacity=int(max(loads)) + 20, dist=d,
                    max_dist=lim, service_time=svc)
    P = oracle_problem(inst)
    lens = np.array([d[t[:-1], t[1:]].sum() for t in tours + tours[:1]], np.float32)
    packed, sizes = pack_tours(tours + [tours[0]], 2 * n)
    with ca.GpuACO(inst, n_ants=ANTS, seed=1, ls_flags=flags, use_graph=False) as g:
        g.init_aco()
        g.set_launch_shape(waves, 16 if waves < 12 else 32, 0, 0, 1)
        g.set_ants(packed, sizes, lens)
        g.local_search()
        got, gsizes, glens = g.ants()
        g.update_statistics()   # folds the per-ant counters into the totals
        evals = g.counters()["ls_evals"]
    total = 0
    for a in range(ANTS):
        t, L, ev = P.local_search(tours[a], flags)
        total += ev
        assert gsizes[a] == len(t), a
        np.testing.assert_array_equal(got[a, : len(t)], t, err_msg=f"ant {a}")
        assert glens[a] == np.float32(L), (a, glens[a], L)
    assert evals == total
