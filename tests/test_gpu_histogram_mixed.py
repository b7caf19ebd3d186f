"""SCC sizes where large SCCs share the whole id range, more and fewer of them
than a block's table of labels holds."""
import numpy as np
import pytest

import ispan_amd as I
from ispan_amd import hiprt as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,k", [(70_000, 1), (70_000, 2), (300_001, 4), (300_001, 100), (300_001, 511),
                                 (300_001, 513), (300_001, 3000), (5_000_000, 3)])
@pytest.mark.parametrize("order", ["by turns", "at random"])
def test_sizes_of_mixed_sccs(V, k, order):
    rng = np.random.default_rng(V + k)
    own = np.arange(V) % k if order == "by turns" else rng.integers(0, k, V)
    by = np.argsort(own, kind="stable")  # a cycle through each SCC's vertices
    ends = np.flatnonzero(np.diff(own[by], append=-1))
    nxt = np.roll(by, -1)
    nxt[ends] = by[np.concatenate([[0], ends[:-1] + 1])]
    # and hubs, or a cycle of V vertices takes V levels
    first = by[np.concatenate([[0], ends[:-1] + 1])]
    hub = first[np.searchsorted(own[first], own)]
    v = np.arange(V)
    src = np.concatenate([by, v, hub]).astype(np.int32)
    dst = np.concatenate([nxt, hub, v]).astype(np.int32)
    a, b = H.DeviceArray(src), H.DeviceArray(dst)
    sizes = np.unique(own, return_counts=True)[1]
    with I.Solver(0) as s:
        dg = s.build_csr(V, src.size, a.ptr, b.ptr)
        a.free()
        b.free()
        try:
            s.bind(dg)
            s.solve()
            bins, summary = s.scc_histogram()
            assert summary == I.get_scc_result(s.labels())
        finally:
            dg.free()
    want = np.zeros(64, np.int64)
    np.add.at(want, np.log2(sizes).astype(int), 1)
    assert np.array_equal(bins, want)
    assert (summary["total"], summary["largest"]) == (sizes.size, sizes.max())
