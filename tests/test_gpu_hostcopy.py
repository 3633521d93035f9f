"""Planes written to the device and read back byte for byte, at sizes around the
pinned ring's: below and at the size from which its helper threads take part, a
slot and the whole ring filled, and one piece more."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import hydrogen as hg

pytestmark = pytest.mark.gpu


def round_trip(n, seed):
    rng = np.random.default_rng(seed)
    a = rng.integers(0, 2**32, (n, n), dtype=np.uint32).view(np.float32)
    b = rng.integers(0, 2**32, (n, n), dtype=np.uint32).view(np.float32)
    with hg.Terrain(n) as t:
        t.write_plane(hg.P_ROCK, a)
        t.write_plane(hg.P_DIRT, b)
        x, y = t.read_plane(hg.P_ROCK), t.read_plane(hg.P_DIRT)
    return np.array_equal(x.view(np.uint32), a.view(np.uint32)) and \
        np.array_equal(y.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n", [8, 504, 512, 520, 720, 728, 1024, 1448, 1456, 2056])
def test_planes_round_trip(n):
    assert round_trip(n, n)


def test_contexts_of_several_threads_copy_at_once():
    ok = [False] * 4

    def work(i):
        ok[i] = all(round_trip(520 + 8 * i, 10 * i + j) for j in range(3))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(ok))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert all(ok)


def test_more_contexts_than_helper_crews():
    """Contexts beyond those that have helpers copy by their own thread."""
    n, a = 520, []
    terrains = [hg.Terrain(n) for _ in range(36)]
    try:
        for i, t in enumerate(terrains):
            a.append(np.random.default_rng(i).random((n, n), dtype=np.float32))
            t.write_plane(hg.P_ROCK, a[-1])
        for t, want in zip(terrains, a):
            assert np.array_equal(t.read_plane(hg.P_ROCK), want)
    finally:
        for t in terrains:
            t.close()
