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
