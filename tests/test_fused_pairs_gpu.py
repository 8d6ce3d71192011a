"""Pull steps taken in pairs (two steps per launch through LDS) against the
one-step kernel, which runs when the steps are asked for one at a time.

Both do the same roundings in the same order, so every comparison is bit for
bit.  Domains: one cell, narrower and wider than a wave, rows and planes that do
not divide into tiles, one or two planes, chunks that end at the last plane.
Cells: walls, spheres, x-face and interior EQU cells (with BOUNCE_BACK or COLLIDE
too), cells without STORE or LOAD."""
from __future__ import annotations

import numpy as np
import pytest

from culbm_amd import Lattice, LatticeConfig, cases
from oracle import pyoracle

pytestmark = pytest.mark.gpu

STORAGE = [("fp32", "nearest"), ("fp16", "nearest"), ("bf16", "nearest"), ("fp16", "stochastic"),
           ("bf16", "stochastic")]


def state(nx, ny, nz, seed=5):
    rng = np.random.default_rng(seed)
    if min(nx, ny, nz) > 2:
        st = cases.channel(nx, ny, nz, u_in=0.06, outlet="zero_gradient" if nx % 2 else "equilibrium")
    else:
        z = np.zeros((nz, ny, nx), np.float32)
        st = cases.State(np.full(z.shape, cases.FLUID, np.uint32), z.copy(), z.copy(), z.copy(), z.copy())
    if min(nx, ny, nz) > 20:
        cases.add_spheres(st, 5, 2.5, 5.0, seed)
    st.rho[...] = 1.0 + rng.uniform(-2e-3, 2e-3, st.shape)
    st.vx += rng.uniform(-1e-2, 1e-2, st.shape).astype(np.float32)
    m = rng.random(st.shape)
    kinds = [cases.EQUILIBRIUM, cases.EQUILIBRIUM | cases.BOUNCE_BACK, cases.EQUILIBRIUM | cases.COLLIDE,
             cases.EQUILIBRIUM | cases.LOAD, cases.COLLIDE | cases.STORE, cases.LOAD | cases.COLLIDE,
             cases.LOAD | cases.BOUNCE_BACK | cases.COLLIDE | cases.STORE]
    for k, flag in enumerate(kinds):
        st.flag[(m > 0.01 * k) & (m < 0.01 * (k + 1))] = flag
    return st


def make(st, **cfg):
    lat = Lattice(LatticeConfig(domain=st.domain, inv_tau=0.7, **cfg))
    lat.set_state(st.flag, st.rho, st.vx, st.vy, st.vz)
    lat.init_ddf("feq")
    return lat


def bits(a):
    return np.where(np.isnan(a), np.uint32(0x7FC00000), a.view(np.uint32))


def singly(lat, n):
    for _ in range(n):
        lat.step(1)


@pytest.mark.parametrize("storage,rounding", STORAGE)
@pytest.mark.parametrize("dim,depth", [((1, 1, 1), 1), ((5, 3, 4), 2), ((33, 40, 1), 1), ((97, 9, 7), 3),
                                       ((130, 17, 2), 2), ((31, 66, 12), 5), ((101, 70, 33), 11),
                                       ((340, 5, 6), 6), ((345, 6, 9), 4), ((700, 4, 5), 5)])
def test_pairs_equal_single_steps(dim, depth, storage, rounding):
    st = state(*dim)
    a = make(st, storage=storage, rounding=rounding)
    b = make(st, storage=storage, rounding=rounding, opt_policy=2, wave_depth=depth)
    singly(a, 7)
    b.step(7)
    assert np.array_equal(bits(a.get_ddf()), bits(b.get_ddf()))
    a.close()
    b.close()


# Domains, and for each storage format from which one on (in this order) the
# library takes pairs on 256 CUs.
AUTO = [(61, 60, 59), (98, 97, 96), (203, 61, 90), (192, 160, 96), (192, 160, 144)]
FIRST_IN_PAIRS = {("fp32", "nearest"): 1, ("fp16", "nearest"): 3, ("bf16", "nearest"): 3, ("fp16", "stochastic"): 4,
                  ("bf16", "stochastic"): 4}


@pytest.mark.parametrize("storage,rounding", STORAGE)
@pytest.mark.parametrize("dim", AUTO)
def test_every_pull_policy_left_to_itself(dim, storage, rounding):
    """Sizes on both sides of where the library starts to take pull steps in pairs:
    one call of several steps, a pending dump and an odd step among them."""
    st = state(*dim)
    pairs = AUTO.index(dim) >= FIRST_IN_PAIRS[storage, rounding]
    a = make(st, storage=storage, rounding=rounding)
    a.step(1)
    a.dump()
    singly(a, 6)
    want = bits(a.get_ddf())
    fields = a.macros()
    a.close()
    for op in (0, 1, 2, 3):
        b = make(st, storage=storage, rounding=rounding, opt_policy=op)
        if op:
            assert (b.info()["launches_per_pass"] == 3) == pairs, op
        b.step(1)
        b.dump_deferred()
        b.step(6)
        assert np.array_equal(want, bits(b.get_ddf())), op
        for x, y in zip(b.macros(), fields):
            assert np.array_equal(bits(x), bits(y)), op
        assert (b.profile_steps(2)["launches"] == 1) == pairs, op
        b.close()


@pytest.mark.parametrize("storage,fmt", [("fp32", np.float32), ("fp16", "fp16"), ("bf16", "bf16")])
def test_pairs_equal_the_oracle(storage, fmt):
    st = cases.config_small(seed=3, n=36)
    lat = make(st, storage=storage, opt_policy=2, wave_depth=9)
    o = pyoracle.Sim(st, 0.7, fmt, scale=lat.info()["storage_scale"])
    o.init_feq()
    lat.step(12)
    o.step(12)
    assert np.array_equal(bits(lat.get_ddf()), bits(o.ddf()))
    lat.close()


@pytest.mark.parametrize("storage,scale", [("fp16", 0.5), ("fp16", 1.0), ("fp16", 2.0 ** 20), ("fp16", 2.0 ** 21),
                                           ("bf16", 2.0 ** -40), ("bf16", 2.0 ** 40)])
def test_explicit_scales(storage, scale):
    """Scales inside and outside the range the pairs compute in."""
    st = state(64, 20, 17)
    a = make(st, storage=storage, storage_scale=scale)
    b = make(st, storage=storage, storage_scale=scale, opt_policy=2, wave_depth=6)
    singly(a, 6)
    b.step(6)
    assert np.array_equal(bits(a.get_ddf()), bits(b.get_ddf()))
    a.close()
    b.close()


@pytest.mark.parametrize("storage", ["fp32", "fp16", "bf16"])
def test_not_a_number_and_infinity(storage):
    """An EQU cell next to a NaN or an infinity keeps its equilibrium."""
    st = cases.channel(40, 24, 20, u_in=0.05)
    ddf = np.random.default_rng(2).normal(0, 1e-3, (27,) + st.shape).astype(np.float32)
    ddf[:, 9, 11, 1:4] = np.nan
    ddf[5, 4, 6, 37] = np.inf
    ddf[6, 5, 6, 2] = -np.inf
    out = []
    for op in (0, 2):
        lat = make(st, storage=storage, storage_scale=0.0 if storage == "fp32" else 1.0, opt_policy=op, wave_depth=7)
        lat.set_ddf(ddf)
        singly(lat, 4) if op == 0 else lat.step(4)
        out.append(lat.get_ddf())
        lat.close()
    assert np.array_equal(bits(out[0]), bits(out[1]))
    assert np.isfinite(out[1][:, 1:-1, 1:-1, 0]).all()
