"""Solves of several hundred iterations: the residual that is left is the true one.

The one-launch and the CSR solves carry s = A p and p.s by recurrence
(cg_resident.hip, cg.hip).  What CG's recursive residual can lose against b - A x is
bounded by the rounding of its updates: about eps ||A|| max ||x_k|| for each of k
iterations (A. Greenbaum, SIAM J. Matrix Anal. Appl. 18, 1997).  The iterates
grow from x = 0 towards x, so max ||x_k|| <= ||x|| up to the last digits, and the
true residual must end below sqrt(tol) + 2 k eps ||A|| ||x||.  Against
the two-reduction iteration (MONO_RESIDENT=0) it may end at most twice as large.

Laplacians plus a storage term of 2e-4 have a condition number of ~6e4 in three
dimensions: several hundred iterations to a relative residual of 1e-13.
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -52


def _system(shape, per_cell):
    """(n, 27) rows, CSR arrays and a function v -> A v of the Laplacian plus storage."""
    nx, ny, nz = shape
    n = nx * ny * nz
    rng = np.random.default_rng(61)
    c = np.arange(n)
    x, y, z = c % nx, c // nx % ny, c // (nx * ny)
    coef = np.zeros((n, 27))
    diag = np.full(n, 2e-4)
    if per_cell:
        diag *= np.exp(rng.normal(0.0, 1.0, n))
    rows, cols, vals = [], [], []
    for slot, ok, off in ((12, x > 0, -1), (14, x < nx - 1, 1), (10, y > 0, -nx), (16, y < ny - 1, nx), (4, z > 0, -nx * ny),
                          (22, z < nz - 1, nx * ny)):
        coef[ok, slot] = -1.0
        diag = diag + ok
        rows.append(c[ok])
        cols.append(c[ok] + off)
        vals.append(np.full(int(ok.sum()), -1.0))
    coef[:, 13] = diag
    rows, cols, vals = np.concatenate(rows + [c]), np.concatenate(cols + [c]), np.concatenate(vals + [diag])
    order = np.lexsort((cols, rows))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    return coef, (rp, cols[order], vals[order]), float(diag.max())


@pytest.mark.parametrize("per_cell", [False, True])
@pytest.mark.parametrize("shape", [(3000, 1, 1), (150, 130, 1), (45, 40, 21)])
def test_true_residual_of_long_solves(oracle, monkeypatch, shape, per_cell):
    import monoalg3d_c_amd as m
    announce(f"long solves {shape} per_cell={per_cell}")
    coef, (rp, col, val), dmax = _system(shape, per_cell)
    n = len(coef)
    x_true = np.random.default_rng(62).normal(size=n) * 80.0
    b = oracle.stencil_apply(shape, coef, x_true)
    tol = 1e-26 * (b @ b)
    left = {}
    for how in ("kernels", "one launch", "csr"):
        monkeypatch.setenv("MONO_RESIDENT", "0" if how == "kernels" else "1")
        if how == "csr":
            x, its, err = m.cg_csr(rp, col, val, b, np.zeros(n), tol=tol, max_its=8000)
        else:
            x, its, err = m.cg_stencil(shape, coef, b, np.zeros(n), tol=tol, max_its=8000)
        r = b - oracle.stencil_apply(shape, coef, x)
        left[how] = float(np.sqrt(r @ r))
        print(f"[long solve] {shape} {how}: {its} iterations, true residual {left[how]:.3e}, recursive {err ** 0.5:.3e}", flush=True)
        assert 300 <= its < 8000 and err <= tol
        assert left[how] <= np.sqrt(tol) + 2 * its * EPS * (2 * dmax) * np.linalg.norm(x)
    assert left["one launch"] <= 2 * left["kernels"]
    assert left["csr"] <= 2 * left["kernels"]
