"""Back-traces that leave the hydro kernels' halo: their cells are listed and
their taps recomputed by 4 lanes each.  Every tile variant of the hydro kernel
and the batch's gives the per-pass result bit for bit, with no such cell, a few
and all of them, also on sides that leave the last tiles nearly empty."""
from __future__ import annotations

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu


def state(n, share):
    """Gentle water; in a share of the cells a large old flux over thin water."""
    rng = np.random.default_rng(n)
    st = np.zeros((hg.NUM_STATE_PLANES, n, n), np.float32)
    st[hg.P_ROCK] = rng.uniform(1.0, 4.0, (n, n))
    st[hg.P_DIRT] = rng.uniform(0.0, 0.5, (n, n))
    st[hg.P_WATER] = rng.uniform(0.5, 1.0, (n, n))
    st[hg.P_SED_ROCK] = rng.uniform(0.0, 1.0, (n, n))
    st[hg.P_SED_DIRT] = rng.uniform(0.0, 1.0, (n, n))
    far = rng.random((n, n)) < share
    st[hg.P_WATER][far] *= 0.02
    for p in (hg.P_FLUX_L, hg.P_FLUX_R, hg.P_FLUX_T, hg.P_FLUX_B):
        st[p][far] = rng.uniform(0.0, 60.0, (n, n))[far]
    return st.astype(np.float32)


def settle(obj):
    obj.set_erosion(hg.erosion_settings())
    obj.set_rain(hg.RAIN_UNIFORM, amount=0.02, seed=1)


@pytest.mark.parametrize("n", [8, 72, 136, 264])
@pytest.mark.parametrize("share", [0.0, 0.01, 1.0])
def test_hydro_variants_with_long_back_traces(n, share):
    st, flags = state(n, share), hg.STEP_DEFAULT
    with hg.Terrain(n) as t:
        settle(t)
        t.write_state(st)
        t.dispatch_grid(2, flags | hg.STEP_PER_PASS)
        want = t.read_state(hg.NUM_STATE_PLANES)
    assert np.isfinite(want).all()
    for v in range(len(hg.tile_variants(hg.KERNEL_HYDRO))):
        print("case", n, share, v, flush=True)
        with hg.Terrain(n) as t:
            settle(t)
            t.set_sweep(-1)
            t.set_tiles(v, 0)
            t.write_state(st)
            t.dispatch_grid(2, flags)
            assert np.array_equal(t.read_state(hg.NUM_STATE_PLANES), want), v
    with hg.Batch([n, 64]) as b:
        settle(b)
        for p in range(hg.NUM_STATE_PLANES):
            b.write_plane(0, p, st[p])
        b.step(2, flags)
        assert np.array_equal(b.read_state(0), want)
