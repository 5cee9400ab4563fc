"""One-launch solves whose blocks give up waiting at any of their exchanges.

With waits of 0 to 30 us (MONO_RESIDENT_WAIT_US, the bound of a kernel's own
wait) some blocks of a solve give up while others have their words, in its first
exchange, in its middle or in its last.  Each such step is solved again by the
kernels of cg.hip, and every step is done once.

Both ways end with r.r <= 1e-16 in every step: within 1e-8 / alpha = 1.4e-7 mV of
the system's solution (the smallest eigenvalue is alpha = 0.07); over 6 steps of a
model that amplifies a difference by less than two per step at most 1e-5 mV.  A step lost or
half solved shows as the step's own change, ~1e-2 mV and more (checked below).
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SHAPE = (100, 90, 4)
STEPS = 6


def _run(m, monkeypatch, precision, seed, resident, wait_us=None):
    monkeypatch.setenv("MONO_RESIDENT", resident)
    if wait_us is None:
        monkeypatch.delenv("MONO_RESIDENT_WAIT_US", raising=False)
    else:
        monkeypatch.setenv("MONO_RESIDENT_WAIT_US", str(wait_us))
    t = m.Tissue(SHAPE, model=m.MODEL_TT2006, precision=precision, tensor=m.iso_tensor(0.00013), cg_tol=1e-16)
    t.v = -85.0 + 100.0 * np.random.default_rng(seed).random(t.n)
    v = [t.v]
    t.step(STEPS - 1)
    v.append(t.v)
    t.step(1)
    v.append(t.v)
    out = v, t.stats
    t.close()
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_steps_left_at_any_exchange_are_solved_again(monkeypatch, precision):
    import monoalg3d_c_amd as m
    announce(f"waits that end early at any exchange, {precision}")
    prec = m.FP64 if precision == "fp64" else m.FP32_REFINE
    for k, wait in enumerate([0, 1, 2, 3, 4, 5, 6, 8, 10, 12, 14, 17, 20, 25, 30]):
        (a0, b0, c0), s0 = _run(m, monkeypatch, prec, 50 + k, "0")
        (a1, b1, c1), s1 = _run(m, monkeypatch, prec, 50 + k, "1", wait)
        assert s1["steps"] == s0["steps"] == STEPS and s1["time"] == s0["time"]
        assert s1["last_cg_error"] <= 1e-16
        np.testing.assert_array_equal(a0, a1)
        assert np.abs(b1 - b0).max() < 1e-5 and np.abs(c1 - c0).max() < 1e-5, wait
        assert np.abs(c0 - b0).max() > 1e-2
