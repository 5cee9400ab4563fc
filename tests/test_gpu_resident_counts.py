"""Which solves run in one launch (mono_tissue_resident_counts).

The comparisons of tests/test_gpu_resident.py pass by themselves where both sides run
the same kernels; here every one of their shapes that fits on the chip has to have its
steps solved in one launch, none with the path switched off, and a run without time to
wait has to have had solves that gave up.  In FP64 a block holds at most 512 x 8 cells,
256 blocks 1,048,576: the two larger shapes are solved by the kernels of cg.hip.
"""
import numpy as np
import pytest

from conftest import announce
from test_gpu_resident import SHAPES

pytestmark = pytest.mark.gpu


def _tissue(m, shape, kind, precision, **more):
    n = int(np.prod(shape))
    rng = np.random.default_rng(21)
    kw = dict(model=m.MODEL_TT2006, precision=precision, tensor=m.iso_tensor(0.00013), cg_tol=1e-16)
    if kind == "holes":
        kw["active"] = (rng.random(n) >= 0.15).astype(np.uint8)
        kw["active"][0] = 1
    elif kind == "factors":
        kw["g_cell"] = np.exp(rng.normal(0.0, 0.3, n))
    elif kind == "layered":
        kw.update(aniso=True, tensor=m.layered_fibre_tensors(shape[2], -60.0, 60.0, 0.00024, 0.000045),
                  tensor_source=m.TENSOR_PER_LAYER)
    elif kind == "fibres":
        th = 0.3 * rng.random(n)
        kw.update(aniso=True, tensor=np.stack([m.fibre_tensor([np.cos(t), np.sin(t), 0.0], 0.00024, 0.000045) for t in th]),
                  tensor_source=m.TENSOR_PER_CELL)
    kw.update(more)
    return m.Tissue(shape, **kw)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind,shape", [(k, s) for k, v in SHAPES.items() for s in v])
def test_steps_are_solved_in_one_launch(monkeypatch, kind, shape, precision):
    import monoalg3d_c_amd as m
    announce(f"one-launch solves counted {kind} {shape} {precision}")
    prec = m.FP64 if precision == "fp64" else m.FP32_REFINE
    monkeypatch.delenv("MONO_RESIDENT", raising=False)
    monkeypatch.delenv("MONO_RESIDENT_WAIT_US", raising=False)
    t = _tissue(m, shape, kind, prec)
    fits = precision == "fp32" or t.n <= 1_048_576
    t.step(3)
    assert t.resident_counts() == (3 if fits else 0, 0)
    t.step(1)
    assert t.resident_counts() == (4 if fits else 0, 0)
    t.close()
    monkeypatch.setenv("MONO_RESIDENT", "0")
    t = _tissue(m, shape, kind, prec)
    t.step(2)
    assert t.resident_counts() == (0, 0)
    t.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_a_run_without_time_to_wait_gives_up(monkeypatch, precision):
    import monoalg3d_c_amd as m
    announce(f"one-launch solves that give up counted {precision}")
    monkeypatch.setenv("MONO_RESIDENT_WAIT_US", "0")
    t = _tissue(m, (128, 130, 1), "holes", m.FP64 if precision == "fp64" else m.FP32_REFINE)
    t.step(60)
    solves, timeouts = t.resident_counts()
    assert timeouts >= 1 and solves + timeouts < 60 and t.stats["steps"] == 60
    t.close()


def test_solves_left_to_the_other_kernels(monkeypatch):
    """Jacobi-preconditioned solves and rows applied from masks."""
    import monoalg3d_c_amd as m
    announce("solves left to the other kernels counted")
    monkeypatch.delenv("MONO_RESIDENT", raising=False)
    holes = (np.random.default_rng(3).random(20 * 14 * 4) >= 0.15).astype(np.uint8)
    for kind, more in (("plain", dict(jacobi=True)), ("layered", dict(active=holes))):
        t = _tissue(m, (20, 14, 4), kind, m.FP64, **more)
        t.step(3)
        assert t.resident_counts() == (0, 0)
        t.close()
