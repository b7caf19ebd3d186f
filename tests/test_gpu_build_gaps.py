"""The edge-list builder with few edges over many rows, compared row by row:
gaps of a few rows, of a wave's, of some pieces and of so many that the pieces
grow, and edge counts around a wave's share of keys."""
import numpy as np
import pytest

import ispan_amd as I
from ispan_amd import hiprt as H
from tests.test_gpu_build import expect

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,m", [
    (40_000_000, 1), (40_000_000, 3), (40_000_000, 200), (33_554_432 + 64 * 8192, 2), (33_554_432 + 4096, 1),
    (8192 * 4096 + 1, 1), (4097 * 3, 3), (5_000_000, 1200), (5_000_000, 40_000),
    (2_000_000, 64 * 2048 - 1), (2_000_000, 64 * 2048), (2_000_000, 64 * 2048 + 1), (2_000_000, 128 * 2048 + 5),
    (500_000, 1024 * 2048 - 64 * 2048), (500_000, 1024 * 2048 + 3),
])
def test_rows_of_gaps(V, m):
    rng = np.random.default_rng(V % 997 + m)
    src, dst = rng.integers(0, V, m), rng.integers(0, V, m)
    a, b = H.DeviceArray(src.astype(np.int32)), H.DeviceArray(dst.astype(np.int32))
    with I.Solver(0) as s:
        dg = s.build_csr(V, m, a.ptr, b.ptr)
        try:
            g = dg.download()
        finally:
            dg.free()
    for got, want in zip((g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj), expect(V, src, dst)):
        assert np.array_equal(got, want)
