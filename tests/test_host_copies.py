"""The host side of copies to and from the device, on a HIP runtime that runs
queued copies as late as the real one may, and fails calls when told to."""
from __future__ import annotations

import pytest

import fakehip


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return fakehip.build(tmp_path_factory.mktemp("fakehip"))


def test_refused_event_leaves_no_error_behind(so):
    """Without an event for a slot the copy takes the runtime's own path; the
    refusal is not the caller's, whose next launch asks for the last error."""
    out = fakehip.run(so, """
        n, a = 512, np.random.default_rng(0).random((512, 512), dtype=np.float32)
        with hg.Terrain(n) as t:
            fake.fake_fail(b"hipEventCreateWithFlags", 1, 2)
            t.write_plane(hg.P_ROCK, a)
            print(fake.fake_last_error())
            t.dispatch_grid(1)
            print(np.array_equal(t.read_plane(hg.P_DIRT), np.zeros((n, n), np.float32)))
        """)
    assert out.split() == ["0", "True"]


@pytest.mark.parametrize("failing", ["hipEventSynchronize", "hipMemcpyAsync"])
@pytest.mark.parametrize("nth", [1, 2, 5])
def test_failed_read_leaves_no_copy_under_way(so, failing, nth):
    """After a read that failed midway, its copies no longer write the slots: what
    is written next arrives whole."""
    out = fakehip.run(so, f"""
        n = 2048
        a, b = (np.random.default_rng(i).random((n, n), dtype=np.float32) for i in range(2))
        with hg.Terrain(n) as t:
            t.write_plane(hg.P_ROCK, a)
            fake.fake_fail(b"{failing}", {nth}, 2)
            try:
                t.read_plane(hg.P_ROCK)
                print("read")
            except hg.HGError:
                print("failed")
            t.write_plane(hg.P_DIRT, b)
            print(np.array_equal(t.read_plane(hg.P_DIRT), b), np.array_equal(t.read_plane(hg.P_ROCK), a))
        """)
    assert out.split() == ["failed", "True", "True"]
