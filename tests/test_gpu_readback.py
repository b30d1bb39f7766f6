"""Readback through the context's two pinned buffers (512 KB each): matrices
whose rows end inside, at and past a buffer, tours with a stride of their
own, and repeated calls.  A copy moves bytes, so everything must be equal."""
import ctypes as C

import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import _lib
from cvrp_aco_ocl_amd.solver import Instance, check, lib

from helpers import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 63, 64, 361, 362, 512, 513, 1024])
def test_pheromone_and_setup_arrays_come_back_whole(n):
    log(f"readback n={n}")
    r = np.random.default_rng(n)
    xy = r.integers(0, 1001, size=(n, 2)).astype(np.float64)
    dem = np.concatenate([[0], r.integers(1, 50, size=n - 1)]).astype(np.int32)
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 500, ca.DIST_NINT)
    with ca.GpuACO(inst, n_ants=5, k=0, seed=1, ls_flags=0, use_graph=False) as g:
        g.init_aco()
        s = g.setup_arrays()
        np.testing.assert_array_equal(s["dist16"], inst.dist.astype(np.uint16))
        np.testing.assert_array_equal(np.take_along_axis(inst.dist, s["nnls"], 1), s["nnd"])
        np.testing.assert_array_equal(s["d0"], inst.dist[0])
        tau = r.uniform(1e-4, 1.0, size=(n, n)).astype(np.float32)
        ti = r.uniform(1e-4, 1.0, size=(n, n)).astype(np.float32)
        for _ in range(2):
            g.set_pheromone(tau, ti)
            got = g.pheromone()
            np.testing.assert_array_equal(got[0], tau)
            np.testing.assert_array_equal(got[1], ti)
            tau, ti = ti, tau


def test_tours_with_a_stride_of_their_own():
    n, m, stride = 400, 700, 1000
    r = np.random.default_rng(5)
    xy = r.integers(0, 1001, size=(n, 2)).astype(np.float64)
    dem = np.concatenate([[0], r.integers(1, 50, size=n - 1)]).astype(np.int32)
    inst = Instance.from_coords(xy[:, 0], xy[:, 1], dem, 500, ca.DIST_NINT)
    with ca.GpuACO(inst, n_ants=m, k=8, seed=1, selection=ca.SEL_KNN, ls_flags=0, use_graph=False) as g:
        g.init_aco()
        g.construct_solutions()
        tours, sizes, lens = g.ants()
        wide = np.full((m + 1, stride), -7, np.int32)
        check(lib.aco_get_ants_at(g.h, 0, wide.ctypes.data_as(C.c_void_p), stride, None, None), "aco_get_ants_at")
        np.testing.assert_array_equal(wide[:, :2 * n], tours)
        assert (wide[:, 2 * n:] == -7).all()
        for a in range(m):
            assert inst.check_solution(tours[a, : sizes[a]])
        with pytest.raises(_lib.AcoError):
            check(lib.aco_get_ants_at(g.h, 0, wide.ctypes.data_as(C.c_void_p), 2 * n - 1, None, None), "aco_get_ants_at")
