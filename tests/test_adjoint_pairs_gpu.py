"""culbm_adjoint with its forward steps in pairs (two steps per launch through LDS)
against the same call with single steps, bit for bit: J, every gradient, dJ/df^0
and the state the context ends in.  Walls, cells without STORE and without LOAD,
both schedules, windows that leave pairs and windows that leave none, and a step
count that continues an earlier run (the stochastic rounding's key)."""
from __future__ import annotations

import numpy as np
import pytest

from culbm_amd import Lattice, LatticeConfig, cases

pytestmark = pytest.mark.gpu

DIM = (33, 21, 19)
KEYS = ("grad_rho", "grad_ux", "grad_uy", "grad_uz", "grad_f0")


@pytest.mark.parametrize("storage,rounding", [("fp32", "nearest"), ("fp16", "nearest"), ("bf16", "nearest"),
                                              ("fp16", "stochastic"), ("bf16", "stochastic")])
@pytest.mark.parametrize("window", [(13, 13), (6, 9), (1, 13)])
@pytest.mark.parametrize("every,slots", [(4, 0), (0, 3), (0, 1)])
def test_pairs_give_the_bits_of_single_steps(storage, rounding, window, every, slots):
    st = cases.channel(*DIM, u_in=0.05, outlet="zero_gradient")
    rng = np.random.default_rng(11)
    st.rho += rng.uniform(-1e-3, 1e-3, st.shape).astype(np.float32)
    m = rng.random(st.shape)
    st.flag[m < 0.02] = cases.LOAD | cases.COLLIDE  # never stored
    st.flag[m > 0.98] = cases.LOAD | cases.BOUNCE_BACK | cases.STORE
    w = rng.uniform(-1, 1, st.shape) * (rng.random(st.shape) < 0.1)
    out = []
    for cfg in (dict(), dict(opt_policy=2, wave_depth=6)):
        lat = Lattice(LatticeConfig(domain=DIM, inv_tau=0.7, storage=storage, rounding=rounding, **cfg))
        lat.set_state(st.flag, st.rho, st.vx, st.vy, st.vz)
        lat.init_ddf("feq")
        lat.step(3)
        out.append((lat.adjoint(w, 13, window, checkpoint_every=every, max_slots=slots, want_f0=True), lat.get_ddf()))
        lat.close()
    (a, fa), (b, fb) = out
    if window != (1, 13) or slots == 1:  # else every state between two is evaluated or kept
        assert b.stats["launches"] < a.stats["launches"]
    assert np.array_equal(fa.view(np.uint32), fb.view(np.uint32))
    assert a.objective == b.objective and a.grad_inv_tau == b.grad_inv_tau
    for k in KEYS:
        x, y = getattr(a, k), getattr(b, k)
        assert np.isfinite(x).all() and np.array_equal(x.view(np.uint8), y.view(np.uint8)), k
    assert np.abs(a.grad_ux).max() > 0 and np.abs(a.grad_f0).max() > 0
