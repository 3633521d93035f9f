"""Copies that take different paths by their size.  Reads of byte counts around the
pinned slots' that are not planes: reference particles of 48 bytes each, one, a
slot less a bit, a slot and a bit, the whole ring and a bit.  First
and later writes below and above the size from which they go through the slots."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 3, 43690, 43691, 174762, 174763])
def test_particles_round_trip(count):
    rng = np.random.default_rng(count)
    want = rng.integers(0, 256, 48 * count, dtype=np.uint8).tobytes()
    with hg.Terrain(64) as t:
        t.ref_particles_init(count)
        t.write_ref_particles((hg.RefParticle * count).from_buffer_copy(want))
        for _ in range(2):
            assert ctypes.string_at(t.read_ref_particles(), 48 * count) == want


@pytest.mark.parametrize("n", [1016, 1024, 2904])
def test_first_and_later_writes(n):
    """Sides around the size from which a plane is written through the slots, from
    the second write on."""
    planes = [np.random.default_rng(i).random((n, n), dtype=np.float32) for i in range(3)]
    with hg.Terrain(n) as t:
        for p in (hg.P_ROCK, hg.P_DIRT, hg.P_WATER):
            t.write_plane(p, planes[p])
        for p in (hg.P_ROCK, hg.P_DIRT, hg.P_WATER):
            assert np.array_equal(t.read_plane(p), planes[p])
