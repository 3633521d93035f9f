"""Droplet counts around a wave's four droplets and a workgroup's 64, on pairs, on the
planes and without allocation: every droplet runs."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [1, 3])
@pytest.mark.parametrize("count", [3, 4, 5, 63, 64, 65])
def test_every_droplet_runs(count, radius):
    """Zero-strength droplets on a slope run 3 steps, or fewer where they leave the
    map at its low side, and change nothing."""
    n, life = 64, 3
    rock = np.broadcast_to((np.arange(n) * 0.01).astype(np.float32)[None, :] + 1.0, (n, n)).copy()
    d = hg.droplet_settings(count=count, max_lifetime=life, erosion=0.0, capacity=0.0, seed=2, brush_radius=radius)
    with hg.Terrain(n) as t, hg.Terrain(8) as out:
        t.write_plane(hg.P_ROCK, rock)
        t.set_droplets(d)
        t.dispatch_particle(1)
        _, steps = t.particle_stats()
        hg.droplets_noalloc(t.device_ptr(hg.P_ROCK), t.device_ptr(hg.P_DIRT), n, d, 0, 1, t.stream(),
                            out.device_ptr(hg.P_VEL_U), out.device_ptr(hg.P_VEL_V))
        t.sync()
        assert int(out.read_plane(hg.P_VEL_V).view(np.uint64).ravel()[0]) == steps
        assert np.array_equal(t.read_plane(hg.P_ROCK), rock) and not t.read_plane(hg.P_DIRT).any()
    assert count <= steps <= life * count and steps >= 0.8 * life * count - 6
