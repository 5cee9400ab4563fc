"""The solve in one launch (cg_resident.hip) against the kernels it replaces.

Both run conjugate gradients with the same stopping rule from the same start,
so the iteration counts agree and the potentials differ by rounding times the
steps' amplification.  In FP64 the rounding of a solve is ~1e-16 relative, on
a potential of 1e2 mV over 20 steps far below 1e-9 mV.  In the mixed precision
both end with an FP64 residual below the tolerance, r.r <= 1e-16, so each is
within 1e-8 / alpha = 1.4e-7 mV of the system's solution (the smallest
eigenvalue is alpha = 0.07), per step; over 20 steps of a model that amplifies a
difference by less than two per step at most 1e-5 mV.  An inner solve may stop
an iteration earlier or later where the FP32 residual is at its threshold.
"""
import os

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def _run(shape, resident, kind, precision, steps, **env):
    import monoalg3d_c_amd as m
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
    env["MONO_RESIDENT"] = "1" if resident else "0"
    try:
        os.environ.update(env)
        t = m.Tissue(shape, **kw)
    finally:
        for k in env:
            os.environ.pop(k)
    t.step(steps)
    out = t.v, t.stats
    t.close()
    return out


# one block and many; tiles that fill their block and tiles cut by the box's
# end; axes of one, two and three cells; 256 and 512 threads and 1, 2, 4, 8 and
# 32 cells per thread (the largest three only with few steps)
SHAPES = {
    "plain": [(300, 1, 1), (1, 700, 1), (1, 1, 65), (2, 2, 2), (40, 1, 7), (33, 17, 9), (64, 64, 1), (100, 80, 20)],
    "holes": [(20, 14, 4), (257, 3, 1), (129, 67, 1), (1100, 1000, 1), (1700, 1500, 1), (120, 100, 33)],
    "factors": [(255, 1, 1), (20, 14, 4), (130, 129, 1), (300, 257, 1), (64, 63, 16)],
    "layered": [(20, 14, 4), (2, 30, 20), (67, 40, 5), (100, 61, 21)],
    "fibres": [(20, 14, 4), (64, 30, 1), (3, 2, 50), (61, 43, 9)],
}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind,shape", [(k, s) for k, v in SHAPES.items() for s in v])
def test_resident_solve_matches_kernel_per_step(kind, shape, precision):
    import monoalg3d_c_amd as m
    announce(f"resident solve {kind} {shape} {precision}")
    prec = m.FP64 if precision == "fp64" else m.FP32_REFINE
    steps = 20 if np.prod(shape) < 500_000 else 4
    v1, s1 = _run(shape, True, kind, prec, steps)
    v0, s0 = _run(shape, False, kind, prec, steps)
    assert s1["steps"] == s0["steps"] and s1["time"] == s0["time"]
    assert np.isfinite(v1).all()
    if precision == "fp64":
        assert s1["inner_iterations_total"] == s0["inner_iterations_total"]
        assert np.abs(v1 - v0).max() < 1e-9
    else:
        assert abs(s1["inner_iterations_total"] - s0["inner_iterations_total"]) <= 0.2 * s0["inner_iterations_total"]
        assert np.abs(v1 - v0).max() < 1e-5
    assert s1["last_cg_error"] <= 1e-16


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_a_wait_that_ends_early_leaves_the_step_to_the_other_kernels(precision):
    """With no time to wait, blocks give up as soon as a word is not there yet:
    those steps are solved by the kernel-per-operation path and the run
    continues, with every step done once."""
    import monoalg3d_c_amd as m
    announce(f"resident solve without waiting, {precision}")
    prec = m.FP64 if precision == "fp64" else m.FP32_REFINE
    shape = (128, 130, 1)
    v1, s1 = _run(shape, True, "holes", prec, 60, MONO_RESIDENT_WAIT_US="0")
    v0, s0 = _run(shape, False, "holes", prec, 60)
    assert s1["steps"] == 60 and s1["time"] == s0["time"]
    assert np.abs(v1 - v0).max() < (1e-7 if precision == "fp64" else 1e-5)


def test_nan_stops_an_enqueued_run_at_its_step():
    """A state that gives a NaN in the first step ends a run of many enqueued
    steps there, as it does when every step is waited for."""
    import monoalg3d_c_amd as m
    announce("NaN stops enqueued steps")
    got = []
    for resident in ("1", "0"):
        os.environ["MONO_RESIDENT"] = resident
        try:
            t = m.Tissue((65, 20, 1), model=m.MODEL_MS2003, tensor=m.iso_tensor(0.00013))
        finally:
            os.environ.pop("MONO_RESIDENT")
        t.step(3)
        v = t.v
        v[77] = np.nan
        t.v = v
        assert t.step(50) == 1
        got.append((t.stats["steps"], t.stats["time"], t.stats["nan_detected"]))
        t.close()
    assert got[0] == got[1] and got[0][0] == 4


def test_two_tissues_in_two_threads():
    """Tissues stepped at the same time from two threads, each on its own
    stream, give what they give one after the other."""
    import threading

    import monoalg3d_c_amd as m
    announce("two tissues in two threads")

    def make(k):
        return m.Tissue((200 + k, 180, 1), model=m.MODEL_TT2006, tensor=m.iso_tensor(0.00013), cg_tol=1e-16)

    alone = []
    for k in range(2):
        t = make(k)
        t.step(100)
        alone.append(t.v)
        t.close()
    both = [make(k) for k in range(2)]
    threads = [threading.Thread(target=t.step, args=(100,)) for t in both]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for t, v in zip(both, alone):
        assert t.stats["steps"] == 100
        assert np.abs(t.v - v).max() < 1e-7
        t.close()
