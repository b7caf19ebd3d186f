"""The grid barrier's records are not cleared between launches: each barrier's
tag goes on from the last one's.  Solves of one context that pass different
numbers of barriers, and barriers of different record sizes, one after
another, give the labels each graph has by itself."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu

GRAPHS = {
    "no_edges": lambda: O.build_csr(70, np.zeros(0, np.int32), np.zeros(0, np.int32)),  # no traversal
    "toy": lambda: G.toy_graph()[0],
    "rmat": lambda: O.rmat(10, 8.0, 3),
    "grid": lambda: O.grid(60, 0.5, 2),          # many levels
    "cycles": lambda: G.cycles_graph(5),         # patterns, WCC and mice
    "chain": lambda: G.cycle_chain(500, 7),      # a second cooperative launch (colouring)
}


@pytest.mark.parametrize("order", ["forward", "backward", "each_twice"])
def test_launches_of_different_lengths_in_turn(order):
    names = list(GRAPHS)
    if order == "backward":
        names = names[::-1]
    elif order == "each_twice":
        names = [n for n in names for _ in range(2)]
    made = {n: GRAPHS[n]() for n in GRAPHS}
    want = {n: O.tarjan(g) for n, g in made.items()}
    with I.Solver(0) as s:
        for rep in range(6):
            for n in names:
                g = made[n]
                s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
                for wcc in (0, 1):
                    s.solve(I.default_params(wcc_mode=wcc))
                    assert np.array_equal(s.labels(), want[n]), (rep, n, wcc)


@pytest.mark.parametrize("wcc", [0, 1, 2])
def test_half_the_blocks_and_all_in_turn(wcc):
    """Graphs at the size up to which half of the blocks are launched, just
    past it, and small ones between, on the same records."""
    made = [O.rmat(17, 4.0, 1), O.grid(363, 0.5, 2), O.rmat(9, 8.0, 3), G.cycle_chain(400, 5)]
    for extra in (0, 1):  # 2^17 vertices, and one isolated vertex more
        V = (1 << 17) + extra
        src = np.repeat(np.arange(made[0].V), np.diff(made[0].fw_beg)).astype(np.int32)
        made.append(O.build_csr(V, src, made[0].fw_adj.astype(np.int32)))
    want = [O.tarjan(g) for g in made]
    with I.Solver(0) as s:
        for _ in range(2):
            for i in (4, 5, 0, 2, 1, 3, 5, 4, 2):
                g = made[i]
                s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
                st = s.solve(I.default_params(wcc_mode=wcc))
                assert st.engine_used == 0
                assert np.array_equal(s.labels(), want[i]), i
