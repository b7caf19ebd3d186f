"""What a context keeps between calls: the builders' scratch up to 1 GiB in
all, given back when something else needs the room, and nothing of a single
graph once a batch is bound or a binding fails."""
import time

import numpy as np
import pytest

import ispan_amd as I
from ispan_amd import hiprt as H

pytestmark = pytest.mark.gpu

MB = 1 << 20


def free():
    """Free device memory, once it has stopped growing: memory is cleared after
    it was freed, and only then counts as free."""
    H.synchronize()
    last, since = H.mem_info()[0], time.monotonic()
    end = since + 10
    while time.monotonic() < min(since + 0.3, end):
        time.sleep(0.02)
        now = H.mem_info()[0]
        if now != last:
            last, since = now, time.monotonic()
    return last


def edges(V, m):
    e = np.random.default_rng(m).integers(0, V, (2, m)).astype(np.int32)
    return H.DeviceArray(e[0]), H.DeviceArray(e[1])


@pytest.mark.parametrize("m", [1_000_000, 60_000_000, 66_900_000])
def test_scratch_of_a_build(m):
    V = 1 << 20
    a, b = edges(V, m)
    with I.Solver(0) as s:
        s.build_csr(V, 1000, a.ptr, b.ptr).free()  # what the first call of a process takes
        before = free()
        s.build_csr(V, m, a.ptr, b.ptr).free()
        assert before - free() <= 1024 * MB + 2 * MB
    a.free()
    b.free()


def test_first_entries_go_with_the_graph():
    V = 50_000_000  # 400 MB of first entries
    beg = H.DeviceArray(np.zeros(V + 1, np.int32))
    small = H.DeviceArray(np.zeros(8, np.int32))
    bad = H.DeviceArray(np.asarray([0, 3, 1, 2], np.int32))
    with I.Solver(0) as s:
        before = free()
        s.bind(I.DeviceGraph(V, 0, beg.ptr, small.ptr, beg.ptr, small.ptr))
        assert before - free() >= 350 * MB
        g = s.gen_rmat(1000, 4.0, 1)
        batch = I.DeviceBatch.from_device([g])
        s.batch_bind(batch)
        assert before - free() <= 100 * MB
        batch.free()
        g.free()
        s.bind(I.DeviceGraph(V, 0, beg.ptr, small.ptr, beg.ptr, small.ptr))
        with pytest.raises(I.IspanError) as e:
            s.bind(I.DeviceGraph(3, 2, bad.ptr, small.ptr, bad.ptr, small.ptr))
        assert e.value.code == -2
        assert before - free() <= 100 * MB
    for d in (beg, small, bad):
        d.free()


def test_kept_scratch_makes_room():
    """With the device nearly full, a solve whose state fits only where the
    scratch of an earlier build lies, and a build whose result does."""
    V = 1 << 20
    a, b = edges(V, 60_000_000)
    n = 10_000_000  # pairs of vertices: 880 MB of solve state
    v = np.arange(n, dtype=np.int32)
    pairs = I.HostGraph(np.arange(n + 1, dtype=np.int32), v ^ 1, np.arange(n + 1, dtype=np.int32), v ^ 1)
    hogs = []
    with I.Solver(0) as s:
        s.build_csr(V, 60_000_000, a.ptr, b.ptr).free()
        b.free()
        a.free()
        a, b = edges(V, 1000)
        try:
            for _ in range(16):
                room = free() - 600 * MB
                if room > 50 * MB:
                    hogs.append(H.malloc(min(room, 32 << 30)))
            assert free() < 700 * MB
            s.upload(pairs)
            st = s.solve()
            assert st.trim2 + st.giant_size == n
            assert np.array_equal(s.labels(), v & ~1)
        finally:
            for h in hogs:
                H.free(h)
    a.free()
    b.free()
