"""J of culbm_adjoint for lists of weighted cells around a wave, a workgroup and
the count from which workgroups take four waves, against the sum over the
dumped velocities of the same run."""
from __future__ import annotations

import numpy as np
import pytest

from culbm_amd import Lattice, LatticeConfig, cases

pytestmark = pytest.mark.gpu

DIM = (67, 53, 41)  # 145,591 cells
STEPS, FIRST = 4, 2


@pytest.mark.parametrize("storage", ["fp32", "fp16"])
@pytest.mark.parametrize("count", [0, 1, 63, 64, 65, 255, 257, 16385, 131071, 131072, 145591])
def test_objective_is_the_weighted_sum_of_velocities(count, storage):
    st = cases.channel(*DIM, u_in=0.05, outlet="zero_gradient")
    rng = np.random.default_rng(count)
    st.rho += rng.uniform(-1e-3, 1e-3, st.shape).astype(np.float32)
    w = np.zeros(st.rho.size)
    w[rng.permutation(w.size)[:count]] = rng.uniform(0.5, 1.5, count)
    w = w.reshape(st.shape)
    made = [Lattice(LatticeConfig(domain=DIM, inv_tau=0.6, storage=storage)) for _ in range(2)]
    for lat in made:
        # every cell dumped; nothing reads the dumped fields back into the flow
        lat.set_state(np.where(st.flag == cases.EQUILIBRIUM, cases.FLUID, st.flag) | cases.DUMP,
                      st.rho, st.vx, st.vy, st.vz)
        lat.init_ddf("feq")
    got = made[0].adjoint(w, STEPS, (FIRST, STEPS)).objective
    want = size = 0.0
    for t in range(1, STEPS + 1):
        made[1].step(1)
        if t >= FIRST:
            made[1].dump()
            term = w * made[1].macros()[1].astype(np.float64)
            want += term.sum()
            size += np.abs(term).sum()
    for lat in made:
        lat.close()
    # both add the same FP64 products, each in its own order
    assert abs(got - want) <= 2 * (STEPS + 64) * 2.0 ** -53 * size + count * STEPS * 2.0 ** -53 * size
