"""The edge-list builder where row numbers come close to the largest int32."""
import numpy as np
import pytest

import ispan_amd as I
from ispan_amd import hiprt as H

pytestmark = pytest.mark.gpu

TOP = 2**31 - 1


def part(ptr, first, n):
    out = np.empty(n, np.int32)
    assert H.rt().hipMemcpy(out.ctypes.data, ptr + 4 * first, out.nbytes, 2) == 0
    return out


@pytest.mark.parametrize("V,last", [(TOP, 1), (TOP, 3), (TOP, 40), (TOP, 4000), (TOP, 5000), (TOP - 1, 30),
                                    (TOP - 62, 70), (TOP - 63, 70), (TOP - 64, 70)])
def test_last_rows(V, last):
    """Edges among the first rows and from V - last on: the rows after the
    last key's, a gap of a few, of a wave's and of more than a piece's rows."""
    rng = np.random.default_rng(last)
    src = np.concatenate([rng.integers(0, 50, 30), V - last - rng.integers(0, 100, 30), [V - last]])
    dst = np.concatenate([rng.integers(0, 50, 30), V - last - rng.integers(0, 100, 30), [0]])
    keep = np.unique(np.stack([src, dst], 1)[src != dst], axis=0)
    a, b = H.DeviceArray(src.astype(np.int32)), H.DeviceArray(dst.astype(np.int32))
    with I.Solver(0) as s:
        g = s.build_csr(V, src.size, a.ptr, b.ptr)
        try:
            assert g.E == len(keep)
            n = 10_000
            for beg, rows in ((g.fw_beg, np.sort(keep[:, 0])), (g.bw_beg, np.sort(keep[:, 1]))):
                for first in (0, V + 1 - n):
                    want = np.searchsorted(rows, np.arange(first, first + n, dtype=np.int64))
                    assert np.array_equal(part(beg, first, n), want)
            assert np.array_equal(part(g.fw_adj, 0, g.E), keep[:, 1])
            assert np.array_equal(part(g.bw_adj, 0, g.E), keep[np.lexsort((keep[:, 0], keep[:, 1]))][:, 0])
        finally:
            g.free()
