"""GPU: the droplet kernel's lane groups at the edges of their work: brushes
smaller and larger than the cells a group has in flight together (32), brushes
cut off by the map's edge, part-filled workgroups, several rounds per
workgroup."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,radius,seed", [(128, 1, 1), (128, 3, 2), (128, 4, 3), (128, 6, 1), (16, 3, 1), (16, 6, 2),
                                           (16, 6, 5), (8, 2, 3), (8, 6, 4)])
def test_single_droplet_any_brush_matches_fp32_oracle(n, radius, seed):
    """One droplet has no concurrency, so it follows the FP32 oracle (the same
    operations in the same order) over a short life, as
    test_single_droplet_matches_fp32_oracle does for the default brush."""
    d = dict(count=1, seed=seed, max_lifetime=12, brush_radius=radius)
    with hg.Terrain(n) as t:
        t.init_fbm(hg.fbm_params(seed=seed, base_freq=1.0 / n, hi=n / 2.0))
        dirt = (np.random.default_rng(seed).random((n, n)) * 0.02).astype(np.float32)
        t.write_plane(hg.P_DIRT, dirt)
        r0 = t.read_plane(hg.P_ROCK)
        t.set_droplets(hg.droplet_settings(**d))
        t.dispatch_particle(1)
        r, dd = t.read_plane(hg.P_ROCK), t.read_plane(hg.P_DIRT)
        ex, steps = t.particle_stats()
    r32, d32 = r0.copy(), dirt.copy()
    ex32 = O.droplets(r32, d32, O.droplet_settings(**d), 0)
    change = max(np.abs(r32 - r0).max(), np.abs(d32 - dirt).max())
    err = max(np.abs(r - r32).max(), np.abs(dd - d32).max())
    print(f"n {n} radius {radius}: steps {steps}, max change {change:.3e}, |gpu-fp32| {err:.3e}")
    assert steps > 0
    assert err <= 1e-5 * max(change, 1e-3)
    assert abs(ex - ex32) <= 1e-5 * max(abs(ex32), 1.0)


@pytest.mark.parametrize("count", [1, 127, 128, 129, 1000])
def test_part_filled_workgroups_run_every_droplet(count):
    """Zero-strength droplets on a slope run their whole life and change nothing."""
    n = 64
    rock = np.broadcast_to((np.arange(n) * 0.01).astype(np.float32)[None, :] + 1.0, (n, n)).copy()
    d = hg.droplet_settings(count=count, max_lifetime=3, erosion=0.0, capacity=0.0, seed=2)
    with hg.Terrain(n) as t:
        t.write_plane(hg.P_ROCK, rock)
        t.set_droplets(d)
        t.dispatch_particle(2)
        _, steps = t.particle_stats()
        assert np.array_equal(t.read_plane(hg.P_ROCK), rock)
        assert not t.read_plane(hg.P_DIRT).any()
    # a droplet ends before 3 steps only where it leaves the map at x < 2
    assert 2 * count <= steps <= 2 * 3 * count and steps >= 0.8 * 2 * 3 * count - 6


def test_noalloc_several_rounds_per_workgroup():
    """More droplets than one round of the largest partials launch: every
    droplet runs and the totals balance the map."""
    n, count = 512, (1 << 21) + 77
    d = hg.droplet_settings(count=count, max_lifetime=2, erosion=0.001, seed=3)
    with hg.Terrain(n) as t, hg.Terrain(8) as out:
        t.init_fbm(hg.fbm_params(seed=5, base_freq=4.0 / n, hi=128.0))
        m0 = t.read_plane(hg.P_ROCK).astype(np.float64).sum()
        hg.droplets_noalloc(t.device_ptr(hg.P_ROCK), t.device_ptr(hg.P_DIRT), n, d, 0, 1, t.stream(),
                            out.device_ptr(hg.P_VEL_U), out.device_ptr(hg.P_VEL_V))
        t.sync()
        m1 = t.read_plane(hg.P_ROCK).astype(np.float64).sum() + t.read_plane(hg.P_DIRT).astype(np.float64).sum()
        ex = float(out.read_plane(hg.P_VEL_U).view(np.float64).ravel()[0])
        steps = int(out.read_plane(hg.P_VEL_V).view(np.uint64).ravel()[0])
    assert abs(m1 + ex - m0) <= 1e-6 * m0
    assert count <= steps <= 2 * count and steps > 1.9 * count


@pytest.mark.parametrize("n", [1768, 1776])
def test_single_droplet_on_pairs_and_on_planes(n):
    """On the larger map pairing the planes does not pay for one droplet of 12
    steps, so it runs on the planes themselves; both follow the FP32 oracle."""
    d = dict(count=1, seed=7, max_lifetime=12)
    with hg.Terrain(n) as t:
        t.init_fbm(hg.fbm_params(seed=7, base_freq=1.0 / 64, hi=32.0))
        dirt = (np.random.default_rng(n).random((n, n)) * 0.02).astype(np.float32)
        t.write_plane(hg.P_DIRT, dirt)
        r0 = t.read_plane(hg.P_ROCK)
        t.set_timing(True)
        t.set_droplets(hg.droplet_settings(**d))
        t.dispatch_particle(1)
        r, dd = t.read_plane(hg.P_ROCK), t.read_plane(hg.P_DIRT)
        ex, steps = t.particle_stats()
        paired = "pair_heights" in t.kernel_stats()
    r32, d32 = r0.copy(), dirt.copy()
    ex32 = O.droplets(r32, d32, O.droplet_settings(**d), 0)
    change = max(np.abs(r32 - r0).max(), np.abs(d32 - dirt).max())
    err = max(np.abs(r - r32).max(), np.abs(dd - d32).max())
    assert paired == (n == 1768)
    assert steps > 0
    assert err <= 1e-5 * max(change, 1e-3)
    assert abs(ex - ex32) <= 1e-5 * max(abs(ex32), 1.0)
