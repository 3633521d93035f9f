"""The adjoint's gather kernels by 512 threads a tile (maps below 768^2) and by
256 (from there on) give the same gradients."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fuse", [0, 15])
@pytest.mark.parametrize("flags", [hg.STEP_DEFAULT, hg.STEP_RAIN, hg.STEP_RAIN | hg.STEP_THERMAL,
                                   hg.STEP_RAIN | hg.STEP_SMOOTH])
def test_both_widths_give_the_same_gradient(flags, fuse):
    """The same terrain on 760^2 and, with 8 more rows and columns, on 768^2: a
    loss away from the added border does not see it within three steps, so the
    gradient is the same (up to the order of the float atomics of back-traces
    beyond one cell, and of the coefficients' double sums)."""
    small, large, steps = 760, 768, 3
    rng = np.random.default_rng(5)
    st = np.zeros((hg.NUM_STATE_PLANES, large, large), np.float32)
    st[hg.P_ROCK] = O.fbm_init(large, O.fbm_params(seed=9, base_freq=1.0 / 12, hi=12.0), np.float32)
    st[hg.P_DIRT] = rng.uniform(0.0, 0.2, (large, large))
    st[hg.P_WATER] = rng.uniform(0.0, 0.05, (large, large))
    st[hg.P_SED_ROCK] = rng.uniform(0.0, 0.05, (large, large))
    g = np.zeros((large, large), np.float32)
    g[:600, :600] = rng.standard_normal((600, 600))       # the other two borders are common
    out = []
    for n in (small, large):
        print("case", n, flags, fuse, flush=True)
        with hg.Terrain(n) as t:
            t.set_erosion(hg.erosion_settings())
            t.set_rain(hg.RAIN_CONSTANT, amount=0.01)
            t.set_adjoint_fusion(fuse)
            t.write_state(np.ascontiguousarray(st[:, :n, :n]))
            t.step = 0
            out.append(t.adjoint_rollout(steps, 2, np.ascontiguousarray(g[:n, :n]), flags))
    (ga, ca), (gb, cb) = out
    scale = np.abs(gb).max()
    assert scale > 0
    assert np.abs(gb[:, small:]).max() == 0 and np.abs(gb[small:, :]).max() == 0
    assert np.abs(ga - gb[:small, :small]).max() <= 1e-6 * scale
    assert np.allclose(ca, cb, rtol=1e-6, atol=1e-12)
