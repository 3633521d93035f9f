"""Which kernels a step launches on small maps, seen by a HIP runtime that
records launches instead of running them (no GPU)."""
from __future__ import annotations

import pytest

import fakehip


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return fakehip.build(tmp_path_factory.mktemp("fakehip"))


@pytest.mark.parametrize("tiles,one_kernel", [(None, True), ((-1, -1), True), ((0, -1), False), ((-1, 0), False),
                                              ((3, 5), False)])
def test_tiles_that_are_set_are_run_on_a_small_map(so, tiles, one_kernel):
    """Untuned maps of up to 648^2 cells run a step as one kernel; a tile variant
    set for either of the two kernels is an explicit choice of these."""
    out = fakehip.run(so, f"""
        for n in (64, 512):
            with hg.Terrain(n) as t:
                if {tiles}:
                    t.set_tiles(*{tiles})
                launched()
                t.dispatch_grid(1)
                step = launched()
                t.adjoint_rollout(2, 2, np.zeros((n, n), np.float32))
                taped = launched()
            for names in (step, taped):
                print(any("k_step_tile" in k for k in names), any("k_fused_hydro" in k for k in names),
                      any("k_fused_thermal" in k or "k_march_thermal" in k for k in names))
        """)
    want = "True False False" if one_kernel else "False True True"
    assert out.split("\n")[:-1] == [want] * 4


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_tile_order_that_is_set_is_the_small_maps_too(so, mode):
    """512^2: 16 tile columns, so each order is taken as it is."""
    out = fakehip.run(so, f"""
        fake.fake_watch(b"k_step_tile", 9)               # its order
        with hg.Terrain(512) as t:
            t.set_xcd_order({mode})
            fake.fake_clear()
            t.dispatch_grid(1)
            print(fake.fake_watched())
            fake.fake_clear()
            t.adjoint_rollout(2, 2, np.zeros((512, 512), np.float32))
            print(fake.fake_watched())
        """)
    assert out.split() == [str(mode)] * 2
