"""Binding a graph: the check counts every violation of both directions, reads
nothing out of the lists, and leaves the first entries the solve needs, at
sizes around a block's and a thread's share, checked or not."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O

pytestmark = pytest.mark.gpu


def graph(V, E, seed):
    rng = np.random.default_rng(seed)
    return O.build_csr(V, rng.integers(0, V, E).astype(np.int32), rng.integers(0, V, E).astype(np.int32))


@pytest.mark.parametrize("V,E", [(1, 0), (1, 1), (5, 0), (255, 300), (256, 2048), (257, 2047), (2049, 2049),
                                 (300000, 100), (70001, 600000), (3, 5000)])
def test_first_entries_come_with_the_check(V, E):
    g = graph(V, E, V + E)
    want = O.tarjan(g)
    with I.Solver(0) as s:
        for validate in (1, 0, 1):
            p = I.default_params(validate=validate)
            s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj), p)
            s.solve(p)
            assert np.array_equal(s.labels(), want)


@pytest.mark.parametrize("offsets,ids", [(1, 0), (0, 1), (7, 0), (0, 300), (5, 40)])
@pytest.mark.parametrize("direction", [0, 1])
def test_violations_are_counted(direction, offsets, ids):
    g = graph(5000, 40000, 3)
    rng = np.random.default_rng(4)
    a = [g.fw_beg.copy(), g.fw_adj.copy(), g.bw_beg.copy(), g.bw_adj.copy()]
    beg, adj = a[2 * direction], a[2 * direction + 1]
    beg[rng.choice(np.arange(1, 5000), offsets, replace=False)] = rng.choice([-5, 1 << 30, 7], offsets)
    adj[rng.choice(len(adj), ids, replace=False)] = rng.choice([-1, 5000, 1 << 30], ids)
    n = sum(int((b[:-1] > b[1:]).sum() + ((x < 0) | (x >= 5000)).sum()) for b, x in ((a[0], a[1]), (a[2], a[3])))
    assert n > 0
    with I.Solver(0) as s:
        with pytest.raises(I.IspanError, match=rf"\({n} violations\)"):
            s.upload(I.HostGraph(*a))
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        s.solve()
        assert np.array_equal(s.labels(), O.tarjan(g))
