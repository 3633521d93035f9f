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


@pytest.mark.parametrize("failing", ["hipEventSynchronize", "hipLaunchKernel"])
@pytest.mark.parametrize("nth", [1, 2, 5])
def test_failed_read_leaves_no_copy_under_way(so, failing, nth):
    """After a read that failed midway, its copies no longer write the slots: what
    is written next arrives whole."""
    out = fakehip.run(so, f"""
        n = 2904                                         # written through the slots too
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


def test_helpers_go_to_who_copies_next(so):
    """32 objects have helper threads at a time; one that came too late gets its
    own at its next copy once another has gone."""
    out = fakehip.run(so, """
        n = 512
        a = np.random.default_rng(0).random((n, n), dtype=np.float32)
        def threads():                                   # ended ones leave the list a moment after they are joined
            time.sleep(0.2)
            return len(os.listdir("/proc/self/task"))
        alone = threads()
        ts = [hg.Terrain(n) for _ in range(33)]
        for t in ts:
            t.write_plane(hg.P_ROCK, a)
            t.read_plane(hg.P_ROCK)
        print(threads() - alone)
        ts.pop(0).close()
        print(threads() - alone)
        ts[-1].read_plane(hg.P_ROCK)
        print(threads() - alone, np.array_equal(ts[-1].read_plane(hg.P_ROCK), a))
        for t in ts:
            t.close()
        print(threads() - alone)
        """)
    assert out.split() == ["96", "93", "96", "True", "0"]


@pytest.mark.parametrize("call", ["write", "read"])
def test_helpers_sleep_while_the_gpu_is_busy(so, call):
    """A copy behind work on the stream waits for it: the helpers' processors are
    others' meanwhile."""
    out = fakehip.run(so, f"""
        n, wait = 2904, 0.05
        a = np.random.default_rng(0).random((n, n), dtype=np.float32)
        with hg.Terrain(n) as t:
            t.write_plane(hg.P_ROCK, a)
            fake.fake_event_delay(int(wait * 1e6))           # 13 of the 17 slots' writes wait, all reads
            cpu = time.process_time()
            t.write_plane(hg.P_DIRT, a) if "{call}" == "write" else t.read_plane(hg.P_ROCK)
            print(time.process_time() - cpu < 13 * wait * 0.5)
        """)
    assert out.split() == ["True"]


@pytest.mark.parametrize("memory", ["hipHostMalloc", "hipMalloc"])
def test_memory_the_runtime_knows_is_copied_by_it(so, memory):
    """A caller's pinned buffer goes over the link without a second copy, and device
    memory is not touched by the host."""
    out = fakehip.run(so, f"""
        n = 1024
        p, a = ctypes.c_void_p(), np.random.default_rng(0).random((n, n), dtype=np.float32)
        fake.{memory}(ctypes.byref(p), ctypes.c_size_t(a.nbytes), 0)
        f = ctypes.cast(p, ctypes.POINTER(ctypes.c_float))
        lib, size = hg.load(), ctypes.c_size_t(n * n)
        with hg.Terrain(n) as t, hg.Batch([n]) as b:
            ctypes.memmove(p, a.ctypes.data, a.nbytes)
            assert lib.hg_write_plane(t.h, hg.P_ROCK, f, size) == 0
            assert lib.hg_batch_write_plane(b.h, 0, hg.P_ROCK, f, size) == 0
            print(fake.fake_direct_copies(), np.array_equal(t.read_plane(hg.P_ROCK), a),
                  np.array_equal(b.read_plane(0, hg.P_ROCK), a))
            for read in (lambda: lib.hg_read_plane(t.h, hg.P_ROCK, f, size),
                         lambda: lib.hg_batch_read_plane(b.h, 0, hg.P_ROCK, f, size)):
                ctypes.memset(p, 0, a.nbytes)
                assert read() == 0
                print(fake.fake_direct_copies(), ctypes.string_at(p, a.nbytes) == a.tobytes())
        """)
    assert out.split() == ["2", "True", "True", "3", "True", "4", "True"]


def test_unknown_pointer_leaves_no_error_behind(so):
    out = fakehip.run(so, """
        a = np.random.default_rng(0).random((1024, 1024), dtype=np.float32)
        with hg.Terrain(1024) as t:
            fake.fake_fail(b"hipPointerGetAttributes", 1, 1)
            t.write_plane(hg.P_ROCK, a)
            fake.fake_fail(b"hipPointerGetAttributes", 1, 1)
            print(np.array_equal(t.read_plane(hg.P_ROCK), a), fake.fake_last_error())
        """)
    assert out.split() == ["True", "0"]


def test_reads_are_not_left_to_a_copy_engine(so):
    """The slots of a read are filled by the library's kernel: an engine may be in
    a state in which it takes 100 us more per copy, at half the rate.  An error
    that the caller's program left behind does not fail it."""
    out = fakehip.run(so, """
        a = np.random.default_rng(0).random((1456, 1456), dtype=np.float32)
        with hg.Terrain(1456) as t:
            t.write_plane(hg.P_ROCK, a)
            fake.fake_clear()
            fake.fake_fail(b"hipMemcpyAsync", 1, 2)
            fake.fake_set_last_error(1)
            print(np.array_equal(t.read_plane(hg.P_ROCK), a), len(launched()), fake.fake_last_error())
        """)
    assert out.split() == ["True", "5", "1"]


@pytest.mark.parametrize("write", ["t.write_plane(hg.P_ROCK, a)", "t.write(hg.CH_HEIGHT, q)",
                                   "b.write_plane(0, hg.P_ROCK, a)"])
def test_first_write_of_a_new_object_needs_no_ring(so, write):
    """It would pay for pinned slots and threads, and gain less than they cost."""
    out = fakehip.run(so, f"""
        n = 1024
        a, q = (np.random.default_rng(i).random(s, dtype=np.float32) for i, s in enumerate([(n, n), (n, n, 4)]))
        threads = len(os.listdir("/proc/self/task"))
        with hg.Terrain(n) as t, hg.Batch([n]) as b:
            for _ in range(2):
                {write}
                print(len(os.listdir("/proc/self/task")) - threads)
        """)
    assert out.split() == ["0", "3"]


@pytest.mark.parametrize("n", [8, 512, 1024])
def test_channel_write_waits_once(so, n):
    """For the copy and the kernel that splits it, also where the kernel fails: the
    caller's memory must not be in use when the call returns."""
    out = fakehip.run(so, f"""
        q = np.random.default_rng(0).random(({n}, {n}, 4), dtype=np.float32)
        with hg.Terrain({n}) as t:
            for _ in range(2):
                t.write(hg.CH_HEIGHT, q)
                fake.fake_clear()
            t.write(hg.CH_HEIGHT, q)
            print(fake.fake_syncs(), launched())
            fake.fake_fail(b"hipLaunchKernel", 1, 2)
            fake.fake_set_last_error(2)                      # what the launch leaves
            try:
                t.write(hg.CH_HEIGHT, q)
            except hg.HGError:
                print(fake.fake_syncs())
        """).split("\n")
    assert out[0].startswith("1 [") and "k_deinterleave_rgba" in out[0]
    assert out[1] == "1"
