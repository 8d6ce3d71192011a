"""culbm_adjoint calls of different sizes on one context, in any order, give the
bits of a context of their own: the workspace kept between calls carries
nothing over."""
from __future__ import annotations

import numpy as np
import pytest

from culbm_amd import Lattice, LatticeConfig, cases

pytestmark = pytest.mark.gpu

KEYS = ("grad_rho", "grad_ux", "grad_uy", "grad_uz")


@pytest.mark.parametrize("storage", ["fp32", "fp16"])
def test_calls_on_one_context_equal_calls_on_their_own(storage):
    dim = (33, 21, 19)
    st = cases.channel(*dim, u_in=0.05, outlet="zero_gradient")
    st.flag[4, 5, 6] = cases.LOAD | cases.COLLIDE  # never stored
    rng = np.random.default_rng(2)

    def lattice():
        lat = Lattice(LatticeConfig(domain=dim, inv_tau=0.6, storage=storage))
        lat.set_state(st.flag, st.rho, st.vx, st.vy, st.vz)
        return lat

    def run(lat, call):
        steps, every, w, f0 = call
        lat.init_ddf("feq")
        return lat.adjoint(w, steps, (1, steps), checkpoint_every=every, want_f0=f0)

    def weights(n):
        w = np.zeros(st.rho.size)
        w[rng.permutation(w.size)[:n]] = rng.uniform(-1, 1, n)
        return w.reshape(st.shape)

    calls = [(5, 2, weights(900), True), (30, 10, weights(70), False), (3, 1, weights(1), False),
             (30, 10, weights(5000), True), (12, 0, weights(0), False)]
    shared = lattice()
    for call in calls + calls[::-1]:
        own = lattice()
        a, b = run(shared, call), run(own, call)
        own.close()
        assert a.objective == b.objective and a.grad_inv_tau == b.grad_inv_tau
        for k in KEYS + (("grad_f0",) if call[3] else ()):
            assert np.array_equal(getattr(a, k), getattr(b, k)), k
    shared.close()
