"""GPU: the one-launch step of small maps (the tile variants of hg_set_sweep,
the default of small maps) at sides around its 32-cell tiles, for the flag
subsets and as the adjoint's taped forward, bit for bit against the per-pass
kernels and the two-kernel step."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu

TILES = [v for v, info in enumerate(hg.tile_variants(hg.KERNEL_SWEEP)) if v >= 10]


def spun_up(n, sweep):
    t = hg.Terrain(n)
    t.set_erosion(hg.erosion_settings())
    t.set_rain(hg.RAIN_UNIFORM, amount=0.02, seed=9)
    t.init_fbm(hg.fbm_params(seed=4, base_freq=1.0 / 24, hi=24.0))
    t.write_plane(hg.P_DIRT, np.random.default_rng(n).random((n, n), dtype=np.float32))
    t.dispatch_grid(2, hg.STEP_DEFAULT | hg.STEP_PER_PASS)
    if sweep is not None:
        t.set_sweep(sweep)
    return t


@pytest.mark.parametrize("n", [8, 24, 32, 40, 64, 104, 264])
@pytest.mark.parametrize("flags", [0, hg.STEP_RAIN, hg.STEP_DEFAULT, hg.STEP_THERMAL, hg.STEP_SMOOTH])
def test_tile_step_equals_per_pass(n, flags):
    with spun_up(n, None) as t:
        t.dispatch_grid(3, flags | hg.STEP_PER_PASS)
        want = t.read_state(hg.NUM_STATE_PLANES)
    for v in TILES:
        with spun_up(n, v) as t:
            t.dispatch_grid(3, flags)
            assert np.array_equal(t.read_state(hg.NUM_STATE_PLANES), want), v


def test_small_map_default_and_explicit_choice():
    """The default (a tile variant while launches are not timed), the two
    kernels set explicitly and the timed default agree; timing sees the two."""
    n, out = 136, []
    for setup in (lambda t: None, lambda t: t.set_sweep(-1), lambda t: t.set_timing(True)):
        with spun_up(n, None) as t:
            assert t.get_sweep() == -1
            setup(t)
            t.dispatch_grid(3)
            names = set(t.kernel_stats())
            out.append(t.read_state(hg.NUM_STATE_PLANES))
    assert {"fused_hydro", "fused_thermal"} <= names and "step_sweep" not in names
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("n,flags", [(72, hg.STEP_DEFAULT), (200, hg.STEP_RAIN | hg.STEP_THERMAL), (72, hg.STEP_RAIN)])
def test_adjoint_tape_from_the_tile_step(n, flags):
    g = (np.random.default_rng(1).random((n, n), dtype=np.float32) - 0.5) / (n * n)
    out = []
    for v in [-1] + TILES:
        with spun_up(n, v) as t:
            gh, gc = t.adjoint_rollout(7, 3, g, flags)
            out.append((gh, gc, t.read_state(hg.NUM_STATE_PLANES)))
    for o in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(o, out[0]))
