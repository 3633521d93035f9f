"""Droplets with a brush of one cell (radius 1), on the planes, on pairs and without
allocation: a single droplet follows the FP32 oracle, and many that meet keep the
mass."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg
import pyoracle as O

pytestmark = pytest.mark.gpu


def terrain(n, seed):
    t = hg.Terrain(n)
    t.init_fbm(hg.fbm_params(seed=seed, base_freq=1.0 / max(n, 32), hi=n / 2.0))
    t.write_plane(hg.P_DIRT, (np.random.default_rng(seed).random((n, n)) * 0.02).astype(np.float32))
    t.set_timing(True)
    return t


@pytest.mark.parametrize("seed", [1, 2, 3])
@pytest.mark.parametrize("n,life,paired", [(8, 511, False), (8, 512, True), (64, 12, False)])
def test_single_droplet_matches_fp32_oracle(n, life, paired, seed):
    d = dict(count=1, seed=seed, max_lifetime=life, brush_radius=1)
    with terrain(n, seed) as t:
        r0, d0 = t.read_plane(hg.P_ROCK), t.read_plane(hg.P_DIRT)
        t.set_droplets(hg.droplet_settings(**d))
        t.dispatch_particle(1)
        r, dd = t.read_plane(hg.P_ROCK), t.read_plane(hg.P_DIRT)
        assert ("pair_heights" in t.kernel_stats()) == paired
    r32, d32 = r0.copy(), d0.copy()
    O.droplets(r32, d32, O.droplet_settings(**d), 0)
    change = max(np.abs(r32 - r0).max(), np.abs(d32 - d0).max())
    # as for the other radii: the same operations in the same order
    assert max(np.abs(r - r32).max(), np.abs(dd - d32).max()) <= 1e-5 * max(change, 1e-3)


@pytest.mark.parametrize("count,paired", [(64, False), (4096, True), (4096, None)])
def test_mass_is_kept(count, paired):
    n = 64
    d = hg.droplet_settings(count=count, max_lifetime=30, brush_radius=1, seed=5)
    with terrain(n, 4) as t, hg.Terrain(8) as out:
        m0 = sum(t.read_plane(p).astype(np.float64).sum() for p in (hg.P_ROCK, hg.P_DIRT))
        if paired is None:
            hg.droplets_noalloc(t.device_ptr(hg.P_ROCK), t.device_ptr(hg.P_DIRT), n, d, 0, 1, t.stream(),
                                out.device_ptr(hg.P_VEL_U), out.device_ptr(hg.P_VEL_V))
            t.sync()
            exported = float(out.read_plane(hg.P_VEL_U).view(np.float64).ravel()[0])
        else:
            t.set_droplets(d)
            t.dispatch_particle(1)
            exported, _ = t.particle_stats()
            assert ("pair_heights" in t.kernel_stats()) == paired
        m1 = sum(t.read_plane(p).astype(np.float64).sum() for p in (hg.P_ROCK, hg.P_DIRT))
    # at most 6 additions a step, each rounded by half an ulp of a height below 64:
    # 4096 * 30 * 6 * 2^-19 = 1.4 at the very worst, its square root's worth in fact
    assert abs(m1 + exported - m0) <= 0.02
