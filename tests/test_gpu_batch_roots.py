"""Batches whose graphs' roots, the whole first level, have lists around the
sizes at which they become work items, are cut into several, and fill the
chunks of the per-graph passes, for few graphs and many, against Tarjan."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O

pytestmark = pytest.mark.gpu


def star(d, seed):
    """A hub of degree d both ways with d vertices, a third of them only out of
    it and a third only into it, ids shuffled; chains hang off some."""
    rng = np.random.default_rng(seed)
    V = 2 * d + 5
    leaf = np.arange(1, d + 1)
    out, back = leaf, np.where(leaf % 3 == 0, leaf, rng.integers(1, d + 1, d))
    e = np.concatenate([np.stack([np.zeros(d, int), out], 1), np.stack([back, np.zeros(d, int)], 1),
                        np.stack([leaf, leaf + d], 1)[::2], np.stack([leaf + d, leaf], 1)[::4]])
    e = rng.permutation(V)[e]
    return O.build_csr(V, e[:, 0].astype(np.int32).copy(), e[:, 1].astype(np.int32).copy())


@pytest.mark.parametrize("degrees", [
    [1], [40], [511, 512, 513], [1023, 1024, 1025, 2047, 2048, 2049], [8191, 8192, 8193, 3],
    list(range(1, 66)), [7, 600] * 150, [1 + i % 40 for i in range(1500)],
], ids=lambda d: f"{len(d)}x{max(d)}")
def test_batch_roots(degrees):
    graphs = [star(d, d + i) for i, d in enumerate(degrees)]
    b = I.DeviceBatch.from_host([I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj) for g in graphs])
    with I.Solver(0) as s:
        s.batch_bind(b)
        for _ in range(2):
            s.batch_solve()
            for g, l in zip(graphs, s.batch_labels()):
                assert np.array_equal(l, O.tarjan(g))
