"""Rows applied from masks against the stored rows, in a box with no symmetry.

The check that enables mask mode compares rows formed from the masks with the assembled
ones; the product that the solves take (aniso_row.h mask_aniso_apply) is compared here:
odd sides, three different cell sides, every cross term, 20 % of the cells inactive.

The potential of the model lies between 0 and 1.  The products differ by ~1e-14 of the
diagonal; both solves, FP64 and FP32+refine, stop at an FP64 residual of
1e-10 ||b||, which leaves at most 1e-10 ||v|| < 1e-8 in any cell (the smallest
eigenvalue is the storage term): over 60 steps of two runs below 1e-6.  A
weight that is wrong by a per cent moves neighbours, which differ by ~0.3, by 1e-4 and more.
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SHAPE = (37, 23, 9)


def _tensors(nz):
    """Per-layer conductivities (xx yy zz xy xz yz), positive definite, all cross terms."""
    rng = np.random.default_rng(71)
    out = np.empty((nz, 6))
    for k in range(nz):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        s = q @ np.diag([0.00024, 0.00012, 0.00006]) @ q.T
        out[k] = s[0, 0], s[1, 1], s[2, 2], s[0, 1], s[0, 2], s[1, 2]
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_mask_products_match_stored_rows(monkeypatch, precision):
    import monoalg3d_c_amd as m
    announce(f"mask products vs stored rows {SHAPE} {precision}")
    n = int(np.prod(SHAPE))
    t6 = _tensors(SHAPE[2])
    assert (np.abs(t6[:, 3:]) > 1e-7).all()
    active = (np.random.default_rng(72).random(n) >= 0.2).astype(np.uint8)
    v0 = np.random.default_rng(73).random(n)
    got = {}
    for mask in ("1", "0"):
        monkeypatch.setenv("MONO_MASK_ROWS", mask)
        monkeypatch.setenv("MONO_RESIDENT", "0")  # the stored rows by the same kernels
        t = m.Tissue(SHAPE, h=(100.0, 140.0, 230.0), model=m.MODEL_MS2003, aniso=True, tensor=t6, tensor_source=m.TENSOR_PER_LAYER,
                     active=active, cg_rel_tol=1e-10, cg_tol=0.0, cg_max_its=500,
                     precision=m.FP64 if precision == "fp64" else m.FP32_REFINE)
        t.v = np.where(active, v0, t.v)
        t.step(60)
        got[mask] = t.v, t.stats
        t.close()
    (v1, s1), (v2, s2) = got["1"], got["0"]
    assert s1["class_operator"] == 3 and s2["class_operator"] == 0
    assert np.isfinite(v1).all() and np.abs(v1 - v2).max() < 1e-6
    assert np.ptp(v1[active != 0]) > 1e-3
