"""CSR conjugate gradient on matrices whose rows take each way through the
product: rows that fit one stretch of products, several stretches per block,
rows longer than a thread adds up (a wave per row), empty and single rows,
block remainders.

The matrices are symmetric with a diagonal that exceeds the sum of the other
entries' magnitudes by 1, so their smallest eigenvalue is at least 1 and a
residual of r.r <= 1e-20 leaves an error of at most 1e-10; the recurrence's
residual differs from the true one by rounding, below 1e-10 here (entries of
order one, at most a few hundred iterations, 1e-16 each).
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def _matrix(kind, n, seed):
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    if kind == "band":     # about 41 entries a row: several stretches per block
        offs = np.arange(1, 21)
        A = sp.diags([rng.normal(size=n - o) for o in offs if o < n], [o for o in offs if o < n], shape=(n, n))
    elif kind == "short":  # up to seven entries, some rows empty off the diagonal
        i, j = rng.integers(0, n, (2, 3 * n))
        A = sp.coo_matrix((rng.normal(size=3 * n), (i, j)), shape=(n, n))
    else:                  # an arrow: one full row and column
        A = sp.lil_matrix((n, n))
        A[0, 1:] = rng.normal(size=n - 1)
    A = sp.triu(A, 1).tocsr()
    A = A + A.T
    d = np.asarray(abs(A).sum(axis=1)).reshape(-1) + 1.0 + rng.random(n)
    A = (A + sp.diags(d)).tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("jacobi", [False, True])
@pytest.mark.parametrize("kind,n", [("short", 1), ("short", 255), ("short", 257), ("short", 5000), ("short", 300_001),
                                    ("band", 30), ("band", 4001), ("arrow", 64), ("arrow", 66), ("arrow", 1500)])
def test_csr_solve_on_rows_of_every_kind(kind, n, jacobi):
    import scipy.sparse.linalg as sl

    import monoalg3d_c_amd as m
    announce(f"csr {kind} n={n} jacobi={jacobi}")
    A = _matrix(kind, n, 11)
    rng = np.random.default_rng(12)
    x = rng.normal(size=n)
    b = A @ x
    got, its, err = m.cg_csr(A.indptr, A.indices, A.data, b, np.zeros(n), tol=1e-20, max_its=2000, jacobi=jacobi)
    assert err <= 1e-20 and its < 2000
    want = x if n > 10_000 else sl.spsolve(A.tocsc(), b)
    assert np.abs(got - want).max() < 2e-10 + 1e-13 * np.abs(want).max()


def test_csr_iteration_cap_and_start_at_the_solution(oracle):
    """Capped solves return the iterate after that many steps, and a start at the
    solution is recognised before any (linear_system_solver.c:95,159-163)."""
    import monoalg3d_c_amd as m
    announce("csr cap")
    A = _matrix("band", 700, 3)
    rng = np.random.default_rng(4)
    b = rng.normal(size=700)
    for cap in (1, 2, 5):
        xr, ir, er = oracle.cg_csr(A.indptr, A.indices, A.data, b, np.zeros(700), 1e-30, cap)
        xg, ig, eg = m.cg_csr(A.indptr, A.indices, A.data, b, np.zeros(700), tol=1e-30, max_its=cap)
        assert ig == ir == cap
        assert np.abs(xg - xr).max() <= 1e-12 * max(1.0, np.abs(xr).max())
        assert eg == pytest.approx(er, rel=1e-9)
    x = m.cg_csr(A.indptr, A.indices, A.data, b, np.zeros(700), tol=1e-26, max_its=500)[0]
    y, its, _ = m.cg_csr(A.indptr, A.indices, A.data, b, x, tol=1e-16)
    assert its == 1 and np.array_equal(x, y)
