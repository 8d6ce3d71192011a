"""Which kernels a configuration takes, on the stand-in runtime (no GPU): the
rules' footprints are those of the buffers that culbm_create allocates."""
from __future__ import annotations

import fakehip


def test_in_place_one_launch_a_step_follows_the_allocated_bytes():
    """FP32 in place, no depth given, domains of 1.6M to 2.4M cells around the
    line, odd widths (padded rows) and even ones (packed) among them."""
    fakehip.run("""
    import random
    rng = random.Random(3)
    dims = [(101, 140, 141), (128, 128, 128), (157, 93, 141), (140, 120, 126), (128, 128, 132), (96, 150, 148)]
    while len(dims) < 24:
        nx, ny = rng.randrange(60, 220), rng.randrange(60, 220)
        nz = round(rng.uniform(185e6, 240e6) / 109 / (nx + 1) / (ny + 1))
        if nz > 40:
            dims.append((nx, ny, nz))
    one = 0
    for nx, ny, nz in dims:
        lat = Lattice(LatticeConfig(domain=(nx, ny, nz), stream_policy=1, opt_policy=3, inner_loop=5))
        populations = lat.info()["device_bytes"] - nx * ny * nz * 20 - (nx * ny * nz + 3) // 4 * 4
        whole = populations + nx * ny * nz <= 227e6
        one += whole
        assert (lat.info()["launches_per_pass"] == 5) == whole, (nx, ny, nz, populations)
        lat.close()
    assert 4 < one < 20
    """)


def test_pull_steps_in_pairs_where_they_measured_faster():
    """Sizes on either side of the line, plain pull steps with no depth given; the
    cache's share does not depend on the rounding mode."""
    fakehip.run("""
    pairs = [("fp32", "nearest", (80, 80, 80)), ("fp32", "nearest", (101, 99, 97)), ("fp32", "nearest", (40, 104, 262)),
             ("fp16", "nearest", (120, 120, 120)), ("fp16", "nearest", (128, 128, 128)), ("fp16", "nearest", (62, 181, 186)),
             ("bf16", "nearest", (144, 128, 120)), ("fp16", "stochastic", (192, 160, 144))]
    plain = [("fp32", "nearest", (72, 72, 72)), ("fp32", "nearest", (84, 84, 44)), ("fp32", "nearest", (64, 64, 64)),
             ("fp16", "nearest", (107, 109, 78)), ("fp16", "nearest", (267, 61, 91)), ("bf16", "nearest", (257, 57, 155)),
             ("fp16", "stochastic", (130, 126, 126)), ("fp16", "stochastic", (203, 170, 119))]
    for want, rows in (("k_fused2", pairs), ("k_pull", plain)):
        for storage, rounding, dim in rows:
            lat = Lattice(LatticeConfig(domain=dim, storage=storage, rounding=rounding))
            fake.fake_clear()
            lat.step(2)
            assert set(launched()) == {want}, (storage, rounding, dim, launched())
            lat.close()
    """)


def test_non_temporal_stores_only_beyond_the_cache():
    """FP32 rows of whole 64-byte blocks: the stores pass the cache by only where it
    holds little of the two buffers."""
    fakehip.run("""
    for dim, nt in [((96, 96, 96), 0), ((112, 96, 96), 0), ((96, 104, 112), 0), ((128, 112, 112), 1), ((160, 136, 136), 1),
                    ((127, 127, 127), 0)]:
        lat = Lattice(LatticeConfig(domain=dim))
        fake.fake_clear()
        lat.step(2)
        (name,) = fake.fake_log().decode().split()
        assert "StoreF32ELb0ELb%dE" % nt in name, (dim, name)
        lat.close()
    """)


def test_the_exported_schedule_is_the_one_that_runs():
    """Launches of a pass against culbm_wave_schedule at the depth the context
    reports: chunked, as deep as the domain and beyond, chosen and given."""
    fakehip.run("""
    from culbm_amd.blocking import wave_schedule
    for dim, storage in (((24, 20, 16), "fp32"), ((24, 20, 16), "fp16"), ((96, 90, 80), "fp32"), ((192, 160, 176), "fp32"),
                         ((192, 160, 176), "fp16"), ((5, 4, 1), "fp32")):
        for sp, op in ((1, 1), (1, 3), (0, 1), (0, 3)):
            for depth in (0, 3, dim[2] - 1, dim[2], dim[2] + 7):
                if sp == 0 and depth == 0:
                    continue  # pull steps left to the library may run in pairs
                for loop in (1, 5):
                    lat = Lattice(LatticeConfig(domain=dim, storage=storage, stream_policy=sp, opt_policy=op,
                                                inner_loop=loop, wave_depth=depth, block_dim=(1, 1, 1), grid_dim=dim))
                    want = wave_schedule(dim[2], lat.info()["wave_depth"], loop)
                    fake.fake_clear()
                    lat.step(loop)
                    what = (dim, storage, sp, op, depth, loop, lat.info())
                    grids = [fake.fake_grid(k) for k in range(len(want) + 1)]
                    assert grids == [-(-(z1 - z0) * dim[0] * dim[1] // 256) for z0, z1, t in want] + [-1], what
                    assert lat.info()["launches_per_pass"] == len(want), what
                    lat.close()
    """)


def test_adjoint_takes_pairs_where_the_context_asks_for_them():
    fakehip.run("""
    dim = (33, 21, 19)
    for kw, pairs in [(dict(), 0), (dict(opt_policy=2), 0), (dict(opt_policy=2, wave_depth=6), 1),
                      (dict(opt_policy=2, wave_depth=6, storage="fp16", storage_scale=0.5), 0)]:
        for every in (0, 4):
            lat = Lattice(LatticeConfig(domain=dim, **kw))
            fake.fake_clear()
            lat.adjoint(np.ones(lat.shape), 20, (20, 20), checkpoint_every=every, max_slots=0 if every else 3)
            assert ("k_fused2" in launched()) == bool(pairs), (kw, every)
            lat.close()
    """)
