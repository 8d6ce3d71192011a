"""Host side of the C ABI on the stand-in runtime (no GPU, kernels do not run):
device memory held and given back, host allocations that fail, the routes and
threads of copies to the host."""
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


def test_kept_workspaces_are_bounded_per_device_and_given_back():
    fakehip.run("""
    GiB = 1 << 30

    def made(dim, steps):
        lat = Lattice(LatticeConfig(domain=dim))
        lat.adjoint(np.ones(lat.shape), steps, (1, steps), checkpoint_every=1)
        return lat

    lats = [made((64, 60, 50), 18) for _ in range(21)]  # about 0.44 GB of workspace each
    own = [lat.info()["device_bytes"] for lat in lats]
    assert sum(own) == fake.fake_bytes()
    base = min(own)
    kept = [b - base for b in own]
    first = sum(k == 0 for k in kept)
    assert 0 < first and kept[:first] == [0] * first and min(kept[first:]) > 0.4e9, kept
    assert 7.5 * GiB < sum(kept) <= 8 * GiB, kept
    # an allocation that only fits once they are given back, by a context that keeps
    # none, by one that does and by a new one
    plain = 27 * 4 * 64 * 60 * 50
    for call in (lats[0].get_ddf, lambda: lats[1].set_ddf(np.zeros((27, 50, 60, 64), np.float32)),
                 lambda: lats[0].init_ddf("feq"), lats[0].moment_sums,
                 lambda: Lattice(LatticeConfig(domain=(16, 16, 16))).close()):
        fake.fake_limit(1 << 40)
        lats[-1].adjoint(np.ones(lats[-1].shape), 18, (1, 18), checkpoint_every=1)
        assert lats[-1].info()["device_bytes"] > base
        fake.fake_limit(fake.fake_bytes())
        call()
        assert lats[-1].info()["device_bytes"] == base
    # one that never fits still fails, and the context goes on
    fake.fake_limit(fake.fake_bytes() + plain // 2)
    try:
        lats[0].get_ddf()
        raise SystemExit("no error")
    except _lib.CulbmError as e:
        assert e.code == _lib.ERR_HIP
    fake.fake_limit(1 << 40)
    lats[0].get_ddf()
    for lat in lats:
        lat.close()
    assert fake.fake_bytes() == 0
    """)


def test_a_failing_host_allocation_never_throws_through_the_c_abi():
    """operator new fails at its first, second, ... call within an entry point until
    the entry point gets through: every outcome is a return code, and the context
    works on."""
    fakehip.run("""
    lib = _lib.lib()

    def outcomes(call):
        codes = []
        for k in range(500):
            fake.fake_fail_new(k)
            codes.append(call())
            used_all = ctypes.c_long.in_dll(fake, "fake_new_left").value >= 0
            fake.fake_fail_new(-1)
            if used_all:
                break
        assert codes[-1] == _lib.OK and set(codes) <= {_lib.OK, _lib.ERR_HIP}, codes
        return codes

    big = Lattice(LatticeConfig(domain=(256, 128, 100)))  # 52 MB of fields: through the ring
    small = Lattice(LatticeConfig(domain=(16, 12, 10)))
    for lat in (small, big):
        fields = [np.random.default_rng(k).random(lat.shape, dtype=np.float32) for k in range(4)]
        lat.set_state(None, *fields)
        out = [np.empty(lat.shape, np.float32) for _ in range(4)]
        ptrs = [_lib.ptr(a) for a in out]
        outcomes(lambda: lib.culbm_get_macros(lat._ctx, *ptrs))
        assert all(np.array_equal(a, b) for a, b in zip(out, fields))
    f = np.empty((27,) + small.shape, np.float32)
    get_ddf, p = lib["culbm_get_ddf"], _lib.ptr(f)  # plain pointers: numpy's own conversions allocate too
    outcomes(lambda: get_ddf(small._ctx, p))
    p = _lib.ptr(fields[0])
    outcomes(lambda: lib.culbm_set_state(small._ctx, None, None, p, None, None))
    outcomes(lambda: lib.culbm_profile_steps(small._ctx, 3, None, None))
    outcomes(lambda: lib.culbm_adjoint_plan(40, 0, 5, None, None))
    w = np.ones(small.shape)
    p = _lib.ptr(w)
    spec, stats = _lib.AdjointSpec(), _lib.AdjointStats()
    spec.nsteps, spec.t_begin, spec.t_end = 6, 1, 6
    codes = outcomes(lambda: lib.culbm_adjoint(small._ctx, ctypes.byref(spec), p, ctypes.byref(stats),
                                               None, None, None, None, None))
    assert len(codes) > 5 and _lib.ERR_HIP in codes
    cfg, held = LatticeConfig(domain=(16, 12, 10)).to_c(), fake.fake_bytes()

    def create():
        h = ctypes.c_void_p()
        rc = lib.culbm_create(ctypes.byref(cfg), ctypes.byref(h))
        assert (rc == _lib.OK) == bool(h.value)
        if h.value:
            lib.culbm_destroy(h)
        assert fake.fake_bytes() == held
        return rc

    assert _lib.ERR_HIP in outcomes(create)
    """)


def test_memory_that_the_runtime_knows_is_copied_to_directly():
    """A caller's pinned (or managed, or device) array takes one copy a field; only
    pageable memory goes through the ring's chunks."""
    fakehip.run("""
    lat = Lattice(LatticeConfig(domain=(256, 128, 100)))  # 13 MB a field
    fields = [np.random.default_rng(k).random(lat.shape, dtype=np.float32) for k in range(4)]
    lat.set_state(None, *fields)
    block = np.empty((4,) + lat.shape, np.float32)
    other = [np.empty(lat.shape, np.float32) for _ in range(4)]
    fake.fake_known(block.ctypes.data, block.nbytes)
    chunk, field = 4 << 20, fields[0].nbytes

    def copy(out):
        fake.fake_clear()
        _lib.check(_lib.lib().culbm_get_macros(lat._ctx, *[_lib.ptr(a) for a in out]), lat._ctx)
        assert all(np.array_equal(a, b) for a, b in zip(out, fields))
        return fake.fake_copies(), fake.fake_largest()

    for _ in range(2):
        assert copy(other) == (16, chunk)
        assert copy(list(block)) == (4, field)
        assert copy(other[:3] + [block[3]]) == (4, field)
    ddf = np.empty((27,) + lat.shape, np.float32)
    fake.fake_known(ddf.ctypes.data, ddf.nbytes)
    fake.fake_clear()
    _lib.check(_lib.lib().culbm_get_ddf(lat._ctx, ddf), lat._ctx)
    assert fake.fake_largest() == ddf.nbytes
    """)


def test_copying_threads_stay_within_the_cpus_the_process_may_use():
    fakehip.run("""
    import os
    lat = Lattice(LatticeConfig(domain=(256, 128, 100)))
    fields = [np.random.default_rng(k).random(lat.shape, dtype=np.float32) for k in range(4)]
    lat.set_state(None, *fields)
    cpus = sorted(os.sched_getaffinity(0))
    for use in (1, min(3, len(cpus)), len(cpus)):
        os.sched_setaffinity(0, set(cpus[:use]))
        before = len(os.listdir("/proc/self/task"))
        fake.fake_clear()
        assert all(np.array_equal(a, b) for a, b in zip(lat.macros(), fields))
        assert fake.fake_threads() - before == min(use, 8), (use, before, fake.fake_threads())
    """)
