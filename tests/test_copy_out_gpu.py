"""Copies to the host: below the size from which they go through the pinned
ring, at it, with chunks that end anywhere, single fields, and two contexts on
two threads at once.  Bytes must arrive unchanged."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from culbm_amd import Lattice, LatticeConfig, _lib, cases

pytestmark = pytest.mark.gpu


def filled(dim, seed=0):
    nx, ny, nz = dim
    rng = np.random.default_rng(seed)
    fields = [rng.random((nz, ny, nx), dtype=np.float32) for _ in range(4)]
    lat = Lattice(LatticeConfig(domain=dim))
    lat.set_state(np.full((nz, ny, nx), cases.FLUID, np.uint32), *fields)
    return lat, fields


@pytest.mark.parametrize("dim", [(5, 7, 3), (127, 129, 31), (128, 128, 32), (127, 129, 33), (256, 256, 80),
                                 (1048577, 1, 1), (257, 131, 127)])
def test_fields_arrive_unchanged(dim):
    lat, fields = filled(dim)
    for _ in range(2):  # the ring serves the smaller ones from the second copy on
        for got, want in zip(lat.macros(), fields):
            assert np.array_equal(got, want)
    one = np.empty(lat.shape, np.float32)
    _lib.check(_lib.lib().culbm_get_macros(lat._ctx, None, None, _lib.ptr(one), None), lat._ctx)
    assert np.array_equal(one, fields[2])
    lat.close()


def test_populations_round_trip():
    lat, _ = filled((101, 97, 23))
    f = np.random.default_rng(1).normal(0, 1e-2, (27,) + lat.shape).astype(np.float32)
    lat.set_ddf(f)
    for _ in range(2):
        assert np.array_equal(lat.get_ddf(), f)
    lat.close()


def test_two_contexts_on_two_threads():
    made = [filled((160, 150, 100), seed) for seed in (3, 4)]
    bad = []

    def read(lat, fields):
        for _ in range(5):
            bad.extend(k for k, (a, b) in enumerate(zip(lat.macros(), fields)) if not np.array_equal(a, b))

    threads = [threading.Thread(target=read, args=m) for m in made]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for lat, _ in made:
        lat.close()


def test_into_pinned_memory():
    lat, fields = filled((160, 150, 100), 5)
    # looked up through the library: the runtime that it runs on
    host_malloc, host_free = _lib.lib()["hipHostMalloc"], _lib.lib()["hipHostFree"]
    block, nbytes = ctypes.c_void_p(), fields[0].nbytes
    assert host_malloc(ctypes.byref(block), ctypes.c_size_t(4 * nbytes), ctypes.c_uint(0)) == 0
    out = np.ctypeslib.as_array(ctypes.cast(block, ctypes.POINTER(ctypes.c_float)), (4,) + lat.shape)
    for _ in range(2):
        out[...] = 0
        _lib.check(_lib.lib().culbm_get_macros(lat._ctx, *[_lib.ptr(a) for a in out]), lat._ctx)
        assert all(np.array_equal(a, b) for a, b in zip(out, fields))
    del out
    lat.close()
    assert host_free(block) == 0
