"""The fused iteration on 16-bit rows, with 4 waves (general relocate) and 8
(packed relocate for long tours), equals the per-phase launches: instances
whose tours are below and above the packed relocate's line, relocate alone
and the full search."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import instances as I

from helpers import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [ca.LS_RELOCATE, ca.LS_2OPT | ca.LS_SWAP | ca.LS_RELOCATE])
@pytest.mark.parametrize("waves", [4, 8])
def test_fused_on_16_bit_rows(waves, flags):
    insts = [I.mixed_1000(3), I.clustered(4), I.uniform_100(5), I.mixed_1000(6).subset(800)]
    log(f"fused row16 waves={waves} flags={flags}")
    out = []
    for shape in ((waves, 16, 0, 0, 1, 1), (waves, 16, 0, 0, 1, 0), (8, 16, 0, 0, 0, 0)):
        with ca.GpuACO(insts, n_ants=16, k=12, seed=9, selection=ca.SEL_KNN, rng=ca.RNG_PHILOX, ls_flags=flags) as g:
            g.init_aco()
            g.set_launch_shape(*shape)
            g.run(3)
            out.append(([g.ants(b) for b in range(len(insts))], [g.pheromone(b) for b in range(len(insts))], g.counters()))
    for ants, phero, counters in out[1:]:
        assert counters == out[0][2]
        for b in range(len(insts)):
            sizes = ants[b][1]
            np.testing.assert_array_equal(out[0][0][b][1], sizes)
            np.testing.assert_array_equal(out[0][0][b][2], ants[b][2])
            for a, size in enumerate(sizes):
                np.testing.assert_array_equal(out[0][0][b][0][a, :size], ants[b][0][a, :size], err_msg=f"{b} {a}")
            for x, y in zip(out[0][1][b], phero[b]):
                np.testing.assert_array_equal(x, y, err_msg=f"instance {b}")
