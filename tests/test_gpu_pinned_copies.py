"""Planes written from and read into a caller's pinned memory, which the copies
reach directly, between the pageable ones of the same object."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 512, 1448])
def test_pinned_planes_round_trip(n):
    rng, lib, size = np.random.default_rng(n), hg.load(), ctypes.c_size_t(n * n)
    hip, p = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p()
    with hg.Terrain(n) as t, hg.Batch([n]) as b:
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(4 * n * n), 0) == 0
        f = ctypes.cast(p, ctypes.POINTER(ctypes.c_float))
        pinned = np.ctypeslib.as_array(f, (n, n))
        for write, read, h in ((lib.hg_write_plane, lib.hg_read_plane, (t.h,)),
                               (lib.hg_batch_write_plane, lib.hg_batch_read_plane, (b.h, 0))):
            for _ in range(2):
                x = rng.random((n, n), dtype=np.float32)
                pinned[:] = x
                assert write(*h, hg.P_ROCK, f, size) == 0
                pinned[:] = 0.0
                assert read(*h, hg.P_ROCK, f, size) == 0
                assert np.array_equal(pinned, x)
                back = t.read_plane(hg.P_ROCK) if len(h) == 1 else b.read_plane(0, hg.P_ROCK)
                assert np.array_equal(back, x)
        assert hip.hipHostFree(p) == 0
