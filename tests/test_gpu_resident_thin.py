"""Rows that reach across an axis of one cell, in the one-launch solve.

A box of one cell along an axis has no neighbour there: whatever coefficient a
row holds for it multiplies nothing (oracle/assembly.c row_apply, the kernels of
cg.hip).  mono_cg_stencil takes any 27-slot rows, so the solve has to give the
oracle's answer for such rows too, stored per cell and as a table.

The rows are strictly dominant (0.02 from each of at most 26 neighbours against a
diagonal of at least 1), so r.r <= tol = 1e-20 leaves at most 1e-10 / 0.48 in x, from
either side: 1e-9 between them.  A coefficient taken for the cell's own would
change the diagonal by 2 % and x by as much.
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SHAPES = [(300, 1, 1), (1, 260, 1), (1, 1, 70), (90, 70, 1), (90, 1, 40), (1, 60, 50), (5000, 1, 1)]


def _rows(shape, kind, rng):
    n = int(np.prod(shape))
    coef = np.zeros((27, n))
    diag = 1.0
    slots = [4, 10, 12, 14, 16, 22] if kind.endswith("7") else [k for k in range(27) if k != 13]
    for k in slots:
        coef[k] = -0.02
    if kind.startswith("cells"):
        diag = 1.0 + rng.random(n)
    coef[13] = diag
    return coef.T


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["table7", "cells7", "table27", "cells27"])
@pytest.mark.parametrize("shape", SHAPES)
def test_rows_across_an_axis_of_one_cell(oracle, shape, kind, precision):
    import monoalg3d_c_amd as m
    announce(f"rows across an axis of one cell {shape} {kind} {precision}")
    n = int(np.prod(shape))
    rng = np.random.default_rng(41)
    coef = _rows(shape, kind, rng)
    b, x0 = rng.normal(size=n), rng.normal(size=n)
    xr, itr, _ = oracle.cg_stencil(shape, coef, b, x0, 1e-20, 200, False)
    x, its, _ = m.cg_stencil(shape, coef, b, x0, tol=1e-20, max_its=200, precision=m.FP64 if precision == "fp64" else m.FP32_REFINE)
    assert np.abs(x - xr).max() < 1e-9
    if precision == "fp64":
        assert abs(its - itr) <= 1
