"""GPU: the reference particle mode's patch loads and corner lanes where they
can go wrong: positions at the map's edges and just below a cell's end (where
adding or subtracting 1 rounds into the next cell), particles leaving, killed,
and beyond the grid.  One dispatch of particles that share no pixel equals the
FP32 oracle bit for bit, as in test_separated_particles_match_fp32_oracle_bitwise."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import hydrogen as hg
import pyoracle as O

pytestmark = pytest.mark.gpu

UNDER = float(np.nextafter(np.float32(3.0), np.float32(0.0)))          # 2.9999998: + 1 rounds to 4
UNDER_BIG = float(np.nextafter(np.float32(33.0), np.float32(0.0)))


@pytest.mark.parametrize("n", [64, 72])
def test_edge_positions_match_fp32_oracle_bitwise(n):
    last = float(n)
    xs = [0.25, 1.0, UNDER, 8.0, 16.5, UNDER_BIG, 40.0, last - 3.0, last - 2.25]
    specs = [(x, 4.0 + 6.0 * j + 0.3, 0.1, -0.05) for j, x in enumerate(xs)]
    specs += [(4.0 + 6.0 * j + 0.3, y, -0.02, 0.1) for j, y in enumerate((0.5, UNDER, last - 1.5, last - 2.75))
              if all(abs(4.0 + 6.0 * j - sx) + abs(y - sy) > 3 for sx, sy, _, _ in specs)]
    specs += [(last + 5.5, 20.5, 0.0, 0.0), (last - 0.5, 45.5, 0.0, 0.0)]
    s = hg.reference_particle_settings(len(specs))
    rng = np.random.default_rng(n)
    with hg.Terrain(n) as t:
        t.init_fbm(hg.fbm_params(seed=3, base_freq=3.0 / n, hi=48.0))
        t.set_erosion(s)
        t.set_ref_particle_dims(n + 16, n + 16)           # positions past the grid stay alive
        t.ref_particles_init(len(specs))
        for p, scale in ((hg.P_FLUX_L, 0.3), (hg.P_FLUX_R, 0.3), (hg.P_DIRT, 0.5), (hg.P_WATER, 1e-5)):
            t.write_plane(p, (rng.random((n, n)) * scale).astype(np.float32))
        parts = (hg.RefParticle * len(specs))()
        for i, (p, (x, y, vx, vy)) in enumerate(zip(parts, specs)):
            p.position[0], p.position[1], p.velocity[0], p.velocity[1] = x, y, vx, vy
            p.iters, p.volume, p.sediment[0], p.sediment[1] = 1, 1.0, 0.01 * i, 0.02
        t.write_ref_particles(parts)
        st = t.read_state(hg.NUM_PLANES)
        t.dispatch_particle_reference(1, should_rain=False, time0=0.5, flags=0)
        got, gst = t.read_ref_particles(), t.read_state(hg.NUM_PLANES)
    op = (O.RefParticle * len(specs))()
    ctypes.memmove(op, parts, ctypes.sizeof(parts))
    os_ = O.ErosionSettings()
    ctypes.memmove(ctypes.byref(os_), ctypes.byref(s), ctypes.sizeof(s))
    O.ref_particle_run(st, op, os_, 1, False, 0.5, 0.0, 0, dims=(n + 16, n + 16))
    for a, b in zip(got, op):
        assert [getattr(a, f) if not hasattr(getattr(a, f), "__len__") else list(getattr(a, f)) for f, _ in a._fields_] \
            == [getattr(b, f) if not hasattr(getattr(b, f), "__len__") else list(getattr(b, f)) for f, _ in a._fields_]
    for k in range(hg.NUM_STATE_PLANES):
        assert np.array_equal(gst[k], st[k]), k
