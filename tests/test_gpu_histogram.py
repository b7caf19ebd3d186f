"""SCC-size histogram at the sizes where its kernels can go wrong: vertex
counts around the four labels a thread loads, the block and the grid, and SCC
sizes around the bins and the sizes counted apart."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O

pytestmark = pytest.mark.gpu


def cycles(sizes, seed):
    """Disjoint cycles of the given sizes over shuffled vertex ids."""
    sizes = np.asarray(sizes, np.int64)
    first = np.cumsum(sizes) - sizes
    V = int(sizes.sum())
    v = np.arange(V)
    g = np.repeat(np.arange(len(sizes)), sizes)
    nxt = first[g] + (v - first[g] + 1) % sizes[g]
    perm = np.random.default_rng(seed).permutation(V)
    return O.build_csr(V, perm[v].astype(np.int32), perm[nxt].astype(np.int32))


@pytest.mark.parametrize("sizes", [
    [1], [2], [3], [4], [1, 4], [2, 3], [3, 3, 1], [4, 4, 4, 1],
    list(range(1, 70)),                       # every bin edge up to 64
    [1] * 1023, [1] * 1024, [1] * 1025,       # a block's labels, and one less and more
    [2] * 700, [1, 2, 3, 4] * 500,
    [5000] + [1] * 4001,                      # one label carried by most vertices
    [300000] + [7] * 20000 + [1] * 100003,    # the whole grid, odd tail
], ids=lambda s: f"{len(s)}x{sum(s)}")
def test_histogram_of_cycles(sizes):
    g = cycles(sizes, len(sizes))
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        s.solve()
        for _ in range(2):  # the size buffer holds the last call's sizes
            bins, summary = s.scc_histogram()
        lab = s.labels()
    want = np.zeros(64, np.int64)
    np.add.at(want, np.log2(np.asarray(sizes)).astype(int), 1)
    assert np.array_equal(bins, want)
    assert summary == I.get_scc_result(lab)
    assert summary["total"] == len(sizes) and summary["largest"] == max(sizes)
