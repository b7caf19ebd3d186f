"""Traversals whose frontier stays narrow for long, then bursts: the sizes at
which a frontier stops being one wave's, one tile, one block's step, or gets a
hub, in both directions, against Tarjan and against level-synchronous solves."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O

pytestmark = pytest.mark.gpu


def bursts(widths, path, tail, seed):
    """A cycle that runs along `path` vertices, through a burst of w parallel
    vertices, along the next path, and so on; from its end a one-way tail of
    `tail` two-vertex cycles.  Vertex ids shuffled."""
    e, v = [], 0
    first = v
    for w in widths:
        e += [(v + i, v + i + 1) for i in range(path)]
        v += path
        e += [(v, v + 1 + i) for i in range(w)] + [(v + 1 + i, v + 1 + w) for i in range(w)]
        v += 1 + w
    e.append((v, first))
    for _ in range(tail):
        e += [(v, v + 1), (v + 1, v + 2), (v + 2, v + 1)]
        v += 2
    e = np.random.default_rng(seed).permutation(v + 1)[np.asarray(e)]
    return O.build_csr(v + 1, e[:, 0].astype(np.int32).copy(), e[:, 1].astype(np.int32).copy())


@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("widths,path,tail", [
    ([1], 300, 0), ([63, 64, 65], 20, 0), ([255, 256, 257], 20, 5), ([511, 512, 513], 20, 5),
    ([1023, 1024, 1025], 9, 0), ([2047, 2048, 2049], 9, 0), ([5000, 3, 700], 40, 300), ([40] * 60, 3, 0),
    ([2, 90, 1, 30], 1500, 4500),
], ids=lambda x: str(x)[:20])
def test_narrow_frontiers(widths, path, tail, flip):
    g = bursts(widths, path, tail, len(widths))
    if flip:
        g = O.Graph(g.bw_beg, g.bw_adj, g.fw_beg, g.fw_adj)
    want = O.tarjan(g)
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        got = {}
        for local in (64, 0):
            st = s.solve(I.default_params(td_local=local))
            assert np.array_equal(s.labels(), want), local
            got[local] = (st.fw_size, st.bw_reach, st.giant_size, st.pivot)
        assert got[64] == got[0]


@pytest.mark.parametrize("ids", ["one place", "two places", "any place"])
@pytest.mark.parametrize("widths,path,tail", [([1, 2, 3], 60, 20), ([60, 20, 60], 30, 5), ([33] * 12, 4, 200)],
                         ids=lambda x: str(x)[:20])
def test_narrow_words_that_share_a_place(widths, path, tail, ids):
    """One wave keeps copies of 256 visited words, by word number modulo 256:
    vertices whose words want the same one or two places, each word with one
    or two of the graph's vertices, and vertices anywhere among many words."""
    g = bursts(widths, path, tail, 7)
    n, V = g.V, 1 << 24
    rng = np.random.default_rng(8)
    if ids == "any place":
        at = rng.choice(V, n, replace=False)
    else:
        k = 1 if ids == "one place" else 2
        word = (np.arange(n) // 2) // k * 256 + (np.arange(n) // 2) % k
        at = rng.permutation(word * 64 + np.arange(n) % 2 * 37)
    V = int(at.max()) + 1
    src = np.repeat(at, np.diff(g.fw_beg)).astype(np.int32)
    g = O.build_csr(V, src, at[g.fw_adj].astype(np.int32))
    want = O.tarjan(g)
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        got = {}
        for local in (64, 0):
            st = s.solve(I.default_params(td_local=local))
            assert np.array_equal(s.labels(), want), local
            got[local] = (st.fw_size, st.bw_reach, st.giant_size, st.pivot)
        assert got[64] == got[0]
