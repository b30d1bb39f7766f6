"""Candidate lists at the edges of the wave-wide row sort: rows around the
part size that lanes sort alone (32) and around one and two passes of 64
elements, few and many equal distances, and rows that are sorted already in
either direction.  Equal to the host builder, row for row."""
import numpy as np
import pytest

import cvrp_aco_ocl_amd as ca

from helpers import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tie", [0, 1])
@pytest.mark.parametrize("shape", ["line", "back", "ties", "spread"])
def test_rows_equal_host_lists(shape, tie):
    insts = []
    for n in (3, 4, 31, 32, 33, 34, 63, 64, 65, 66, 129, 130, 257, 2050):
        r = np.random.default_rng(n)
        x = {"line": np.arange(n), "back": n - np.arange(n), "ties": r.integers(0, 4, size=n),
             "spread": r.integers(0, 10 ** 6, size=n)}[shape].astype(np.float64)
        y = np.zeros(n) if shape in ("line", "back") else r.permutation(x)
        insts.append(ca.Instance.from_coords(x, y, np.concatenate([[0], np.ones(n - 1)]).astype(np.int32), n, ca.DIST_NINT))
    widths = [it.n - 2 for it in insts]
    got = ca.Instance.nn_lists_batch(insts, widths, tie)
    for it, w, g in zip(insts, widths, got):
        log(f"rows {shape} tie={tie} n={it.n}")
        np.testing.assert_array_equal(g, it.nn_lists(w, tie), err_msg=f"n={it.n}")
