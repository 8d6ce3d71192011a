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
