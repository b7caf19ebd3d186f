"""Edge list -> CSR pair on the device against numpy, at the sizes where its
kernels can go wrong: ids that just fit or just pass a 32-bit key, edge counts
around a wave's chunk of keys, rows around a block's, nothing left to keep."""
import numpy as np
import pytest

import ispan_amd as I
from ispan_amd import hiprt as H

pytestmark = pytest.mark.gpu


def expect(V, src, dst):
    key = np.unique(src.astype(np.int64) * V + dst)
    s, d = key // max(V, 1), key % max(V, 1)
    s, d = s[s != d], d[s != d]
    beg = np.searchsorted(s, np.arange(V + 1))
    o = np.lexsort((s, d))
    return beg, d, np.searchsorted(d[o], np.arange(V + 1)), s[o]


def edges(V, m, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "same":        # one edge, many times
        return np.full(m, V - 1), np.zeros(m, np.int64)
    if kind == "loops":       # nothing is kept
        s = rng.integers(0, V, m)
        return s, s
    if kind == "ends":        # rows only at both ends of the id range
        return rng.choice([0, V - 1], m), rng.integers(0, V, m)
    if kind == "skewed":
        return (rng.random((2, m)) ** 3 * V).astype(np.int64)
    return rng.integers(0, V, (2, m))


@pytest.mark.parametrize("V,m", [
    (1, 5), (2, 1), (2, 3000), (3, 1023), (255, 1024), (256, 1025), (257, 4097), (65535, 5000), (65536, 200001),
    (65537, 200001), (1 << 20, 300000), ((1 << 20) + 1, 1 << 20), (300000, 3_000_001), (1 << 24, 70000),
    (2_000_000_000, 1000),
])
@pytest.mark.parametrize("kind", ["uniform", "skewed", "ends", "same", "loops"])
def test_build_csr(V, m, kind):
    if V > 1 << 24 and kind != "uniform":
        pytest.skip("one layout is enough at this many rows")
    src, dst = edges(V, m, kind, V % 1000 + m)
    a, b = H.DeviceArray(src.astype(np.int32)), H.DeviceArray(dst.astype(np.int32))
    with I.Solver(0) as s:
        dg = s.build_csr(V, m, a.ptr, b.ptr)
        try:
            if V > 1 << 24:  # the offsets are too long to compare one by one here
                assert dg.E == len(np.unique(src * V + dst)) - np.sum(np.unique(src[src == dst]).size)
                return
            g = dg.download()
        finally:
            dg.free()
    for got, want in zip((g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj), expect(V, src, dst)):
        assert np.array_equal(got, want)


def test_build_csr_rejects_an_id_outside():
    for s, d in ((0, 7), (7, 0), (-1, 0), (0, -1)):
        a, b = H.DeviceArray(np.asarray([0, s], np.int32)), H.DeviceArray(np.asarray([1, d], np.int32))
        with I.Solver(0) as S, pytest.raises(I.IspanError) as e:
            S.build_csr(7, 2, a.ptr, b.ptr)
        assert e.value.code == -2


@pytest.mark.parametrize("kind", ["uniform", "skewed"])
@pytest.mark.parametrize("V", [40000, 70000])
@pytest.mark.parametrize("m", [(1 << 18) - 1, 1 << 18, (1 << 18) + 1, 262143 + 8192, 600_000])
def test_build_csr_where_the_sorts_change(V, m, kind):
    """Around the size from which keys are sorted by radix passes, where the
    second sort, of the fewer kept keys, still merges."""
    test_build_csr(V, m, kind)
