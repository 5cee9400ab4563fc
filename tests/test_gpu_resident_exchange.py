"""Solves in one launch right after solves that gave their memory back.

Every block-to-block word of cg_resident.hip carries the number of its exchange,
counted from one in each workspace.  A workspace made where another has just been
released must not find the other's first words there: short solves of different
systems, one after the other, each against the kernels of cg.hip.

In FP64 both paths run the same iteration up to the order of their sums: over
3e4 terms a sum differs by ~1e-13 of itself, an iterate of three iterations by a
few times that of its largest value, so by less than 1e-11.  With FP32 inner
solves a correction is rounded to 6e-8 of itself at each of a few dozen
operations, less than 1e-5 of the largest value.  A stale sum changes alpha by
its own size.
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SHAPE = (64, 50, 10)


def _solve(m, monkeypatch, resident, precision, coef, b, x0, max_its):
    monkeypatch.setenv("MONO_RESIDENT", "1" if resident else "0")
    return m.cg_stencil(SHAPE, coef, b, x0, tol=1e-30, max_its=max_its, precision=precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_short_solves_of_different_systems(monkeypatch, precision):
    import monoalg3d_c_amd as m
    announce(f"short solves of different systems, {precision}")
    prec, rel = (m.FP64, 1e-11) if precision == "fp64" else (m.FP32_REFINE, 1e-5)
    n = int(np.prod(SHAPE))
    coef, a = m.assemble(SHAPE, tensor=m.iso_tensor(0.00013))
    rng = np.random.default_rng(31)
    systems = [(rng.normal(size=n) * a * 10.0 ** rng.uniform(-2, 3), rng.normal(-60.0, 20.0, n), k) for _ in range(4) for k in (1, 2, 3)]
    want = [_solve(m, monkeypatch, False, prec, coef, b, x0, k) for b, x0, k in systems]
    for (b, x0, k), (xw, iw, ew) in zip(systems, want):
        x, its, err = _solve(m, monkeypatch, True, prec, coef, b, x0, k)
        assert its == iw, k
        assert np.abs(x - xw).max() <= rel * max(np.abs(xw).max(), np.abs(x0).max()), k


def test_tissues_closed_after_their_first_step(monkeypatch):
    import monoalg3d_c_amd as m
    announce("tissues closed after their first step")
    n = int(np.prod(SHAPE))
    got = {}
    for resident in ("0", "1"):
        monkeypatch.setenv("MONO_RESIDENT", resident)
        rng = np.random.default_rng(32)
        for k in range(6):
            t = m.Tissue(SHAPE, model=m.MODEL_MS2003, tensor=m.iso_tensor(0.00013), cg_tol=1e-16)
            t.step(1)  # a uniform tissue: converged after an iteration
            t.v = rng.random(n)
            t.step(1)
            got[resident, k] = t.v
            t.close()
    for k in range(6):
        assert np.abs(got["1", k] - got["0", k]).max() < 1e-7  # r.r <= 1e-16, smallest eigenvalue 0.07
