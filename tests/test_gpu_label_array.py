"""Where a caller's label array may lie: over the bound graph's own arrays (the
solve is done with them by the time the labels come), and not past the end of
its allocation."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O
from ispan_amd import hiprt as H
from tests import graphs as G

pytestmark = pytest.mark.gpu

GRAPHS = {
    "rmat": lambda: O.rmat(14, 8.0, 3),
    "sparse": lambda: O.rmat(15, 3.0, 4),
    "grid": lambda: O.grid(90, 0.5, 2),
    "cycles": lambda: G.cycles_graph(5),
    "chain": lambda: G.cycle_chain(500, 7),
}


@pytest.mark.parametrize("which", [0, 1, 2, 3], ids=["fw_beg", "fw_adj", "bw_beg", "bw_adj"])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_labels_over_the_graph(name, which):
    g = GRAPHS[name]()
    want = O.tarjan(g)
    host = [np.asarray(x, np.int32) for x in (g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj)]
    if host[which].size < g.V:
        pytest.skip("the array is shorter than the labels")
    with I.Solver(0) as s:
        for kw in ({}, {"wcc_mode": 1}, {"wcc_mode": 2}, {"engine": 1}):
            dev = [H.DeviceArray(x) for x in host]
            s.bind(I.DeviceGraph(g.V, g.fw_adj.size, *[d.ptr for d in dev]))
            s.solve(I.default_params(**kw), dev[which].ptr)
            assert np.array_equal(dev[which].download()[:g.V], want), kw
            for k, d in enumerate(dev):
                if k != which:
                    assert np.array_equal(d.download(), host[k])
                d.free()


def test_too_short_an_array_is_refused():
    g = O.rmat(8, 6.0, 1)
    want = O.tarjan(g)
    out = H.DeviceArray(np.full(g.V, -7, np.int32))
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        with pytest.raises(I.IspanError) as e:
            s.solve(I.default_params(), out.ptr + 4)
        assert e.value.code == -4
        assert (out.download() == -7).all()
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))  # nothing is left of the error
        s.solve(I.default_params(), out.ptr)
        assert np.array_equal(out.download(), want)
    out.free()
