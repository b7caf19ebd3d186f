"""Labels into a caller's device array: at every alignment, with and without
vertices left for later launches, for odd sizes, and apart from the context's
own copy."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O
from ispan_amd import hiprt as H
from tests import graphs as G

pytestmark = pytest.mark.gpu

GRAPHS = {
    "one": lambda: O.build_csr(1, np.zeros(0, np.int32), np.zeros(0, np.int32)),
    "rmat": lambda: O.rmat(12, 8.0, 3),
    "grid": lambda: O.grid(61, 0.5, 2),
    "cycles": lambda: G.cycles_graph(5),    # size-2/3 patterns, WCCs and mice
    "random": lambda: G.random_graph(11),
    "chain": lambda: G.cycle_chain(500, 7),  # the colouring method
}


@pytest.mark.parametrize("name", list(GRAPHS))
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_labels_into_a_callers_array(name, offset):
    g = GRAPHS[name]()
    want = O.tarjan(g)
    out = H.DeviceArray(np.full(g.V + 8, -7, np.int32))
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        for kw in ({}, {"wcc_mode": 2}, {"trim_times": 0}, {"engine": 1}):
            out.upload(np.full(g.V + 8, -7, np.int32))
            s.solve(I.default_params(**kw), out.ptr + 4 * offset)
            got = out.download()
            assert np.array_equal(got[offset:offset + g.V], want), kw
            assert (got[:offset] == -7).all() and (got[offset + g.V:] == -7).all()
            out.upload(np.full(g.V + 8, -7, np.int32))  # the context keeps its own
            assert np.array_equal(s.labels(), want)
