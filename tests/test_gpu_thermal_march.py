"""GPU: the marching thermal kernel (the last HG_KERNEL_THERMAL variant) where
its strips and row segments end: sides around multiples of the 116 columns a
wave writes and of its row segments, every flag combination, the adjoint's
tape, batches.  All of it equals the per-pass kernels bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu

MARCH = len(hg.tile_variants(hg.KERNEL_THERMAL)) - 1


def spun_up(n, seed=3):
    t = hg.Terrain(n)
    t.set_erosion(hg.erosion_settings())
    t.set_rain(hg.RAIN_UNIFORM, amount=0.02, seed=seed)
    t.init_fbm(hg.fbm_params(seed=seed, base_freq=1.0 / 24, hi=24.0))
    t.write_plane(hg.P_DIRT, np.random.default_rng(seed).random((n, n), dtype=np.float32))
    t.dispatch_grid(2, hg.STEP_DEFAULT | hg.STEP_PER_PASS)
    return t


@pytest.mark.parametrize("n", [8, 56, 64, 112, 120, 232, 240, 352, 776])
@pytest.mark.parametrize("flags", [hg.STEP_DEFAULT, hg.STEP_THERMAL, hg.STEP_SMOOTH, hg.STEP_RAIN | hg.STEP_SMOOTH])
def test_march_equals_per_pass(n, flags):
    with spun_up(n) as a, spun_up(n) as b:
        a.set_tiles(-1, MARCH)
        a.dispatch_grid(3, flags)
        b.dispatch_grid(3, flags | hg.STEP_PER_PASS)
        x, y = a.read_state(hg.NUM_STATE_PLANES), b.read_state(hg.NUM_STATE_PLANES)
    assert np.isfinite(x).all()
    assert np.array_equal(x, y)


@pytest.mark.parametrize("n", [120, 352])
@pytest.mark.parametrize("flags", [hg.STEP_THERMAL | hg.STEP_SMOOTH, hg.STEP_THERMAL])
def test_march_equals_tiles_beside_infinite_heights(n, flags):
    """The thermal passes alone (after an iteration of no droplets) on a map with
    single infinities, pairs and a plateau of them, and cells that are no number:
    the same cells are infinite or no number as with the tile kernel, and the
    others are equal."""
    rng, out = np.random.default_rng(n), []
    rock = rng.random((n, n), dtype=np.float32) * 24
    dirt = rng.random((n, n), dtype=np.float32)
    rock[20, 30] = rock[60, 57] = rock[60, 58] = rock[n - 1, 0] = np.inf
    rock[80:90, 50:66] = np.inf
    rock[40, 90], dirt[100, 20], rock[8, 100] = -np.inf, np.inf, np.nan
    dirt[30:33, 3:6] = -np.inf
    for v in (0, MARCH):
        with hg.Terrain(n) as t:
            t.set_erosion(hg.erosion_settings())
            t.write_plane(hg.P_ROCK, rock)
            t.write_plane(hg.P_DIRT, dirt)
            t.set_droplets(hg.droplet_settings(count=0))
            t.set_tiles(-1, v)
            t.dispatch_particle(1, flags)
            out.append(t.read_state(hg.NUM_STATE_PLANES)[:2])
    assert not np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1], equal_nan=True)


def test_march_records_the_adjoint_tape():
    n, out = 232, []
    g = (np.random.default_rng(1).random((n, n), dtype=np.float32) - 0.5) / (n * n)
    for v in (0, MARCH):
        with spun_up(n) as t:
            t.set_tiles(-1, v)
            gh, gc = t.adjoint_rollout(6, 4, g)
            out.append((gh, gc, t.read_state(hg.NUM_STATE_PLANES)))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("flags", [hg.STEP_DEFAULT, hg.STEP_SMOOTH])
def test_march_in_a_batch(flags):
    sides = [8, 120, 256, 440]
    states = []
    for v in (0, MARCH):
        with hg.Batch(sides) as b:
            b.set_rain(hg.RAIN_UNIFORM, amount=0.02, seed=5)
            b.set_erosion(hg.erosion_settings())
            for i, n in enumerate(sides):
                b.init_fbm(i, hg.fbm_params(seed=i + 1, base_freq=1.0 / 24, hi=24.0))
            b.set_tiles(-1, v)
            b.step(3, flags)
            b.set_persistent(True)
            b.step(1, flags)
            states.append([b.read_state(i) for i in range(len(sides))])
    for x, y in zip(*states):
        assert np.array_equal(x, y)


def test_march_per_terrain_launches_of_a_batch():
    """A batch's terrains launched one by one, eagerly and from a graph, take row
    segments of their own."""
    sides, flags, states = [8, 120, 256, 1032], hg.STEP_DEFAULT, []
    for per_terrain in (0, hg.STEP_PER_TERRAIN):
        with hg.Batch(sides) as b:
            b.set_rain(hg.RAIN_UNIFORM, amount=0.02, seed=5)
            b.set_erosion(hg.erosion_settings())
            for i, n in enumerate(sides):
                b.init_fbm(i, hg.fbm_params(seed=i + 1, base_freq=1.0 / 24, hi=24.0))
            b.set_tiles(-1, MARCH)
            b.step(2, flags | per_terrain)
            b.capture(2, flags | per_terrain)
            for _ in range(3):
                b.run()
            b.sync()
            states.append([b.read_state(i) for i in range(len(sides))])
    for x, y in zip(*states):
        assert np.array_equal(x, y)
