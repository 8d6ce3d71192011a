"""Host side of the C ABI on the stand-in runtime (no GPU, kernels do not run):
device memory held and given back."""
from __future__ import annotations

import fakehip


def test_device_bytes_counts_the_kept_workspace():
    fakehip.run("""
    lat = Lattice(LatticeConfig(domain=(24, 20, 16)))
    base = lat.info()["device_bytes"]
    assert base == fake.fake_bytes()
    r = lat.adjoint(np.ones(lat.shape), 5, (1, 5))
    assert fake.fake_bytes() > base  # the workspace is kept
    assert lat.info()["device_bytes"] == fake.fake_bytes()
    lat.close()
    assert fake.fake_bytes() == 0
    """)


def test_memory_cap_bounds_a_workspace_kept_from_an_earlier_call():
    fakehip.run("""
    lat = Lattice(LatticeConfig(domain=(24, 20, 16)))
    w = np.ones(lat.shape)
    base = fake.fake_bytes()
    lat.adjoint(w, 40, (1, 40), checkpoint_every=1)
    cap = (fake.fake_bytes() - base) // 4
    assert lat.adjoint(w, 40, (1, 40), mem_cap=cap).stats["device_bytes"] <= cap
    assert fake.fake_bytes() - base <= cap
    held = fake.fake_bytes()  # a later call without a cap, or one that fits, takes what is there
    lat.adjoint(w, 2, (1, 2))
    lat.adjoint(w, 40, (1, 40), mem_cap=cap)
    assert fake.fake_bytes() == held
    lat.close()
    """)
