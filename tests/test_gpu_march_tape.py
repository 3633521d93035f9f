"""GPU: the marching thermal kernel as the taped forward of the adjoint, on sides on
which it runs without being asked to be and beyond those of one-kernel steps, against
the tile kernel's tape: the same gradients and final state."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu

MARCH = len(hg.tile_variants(hg.KERNEL_THERMAL)) - 1


@pytest.mark.parametrize("n,flags,thermal", [(776, hg.STEP_DEFAULT, MARCH), (776, hg.STEP_THERMAL, MARCH),
                                             (776, hg.STEP_SMOOTH, MARCH), (2048, hg.STEP_DEFAULT, None)])
def test_gradients_from_the_marching_tape(n, flags, thermal):
    out = []
    g = (np.random.default_rng(1).random((n, n), dtype=np.float32) - 0.5) / (n * n)
    for v in (2, thermal):
        with hg.Terrain(n) as t:
            t.set_erosion(hg.erosion_settings())
            t.set_rain(hg.RAIN_UNIFORM, amount=0.02, seed=3)
            t.init_fbm(hg.fbm_params(seed=3, base_freq=1.0 / 24, hi=24.0))
            t.write_plane(hg.P_DIRT, np.random.default_rng(n).random((n, n), dtype=np.float32))
            t.dispatch_grid(2, hg.STEP_DEFAULT | hg.STEP_PER_PASS)
            t.set_sweep(-1)
            if v is not None:
                t.set_tiles(-1, v)
            assert t.get_tiles()[1] == (MARCH if v is None else v)
            gh, gc = t.adjoint_rollout(3, 2, g, flags)
            out.append((gh, gc, t.read_state(hg.NUM_STATE_PLANES)))
    assert np.isfinite(out[0][0]).all() and out[0][0].any()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
