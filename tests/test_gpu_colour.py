"""The colouring method where a block takes what is left alone (at most 1024
vertices) and where all blocks do, from the first round or a later one, with
lists around the four entries it reads at a time, against Tarjan."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O

pytestmark = pytest.mark.gpu


def cycles(n, links, seed, shuffle):
    """n vertices in cycles of 4 to 7 (so no size-2 or size-3 pattern), each
    with an edge to the next cycle and `links` more to later ones: one weakly
    connected piece of many SCCs; a first cycle with chords is the pivot's."""
    rng = np.random.default_rng(seed)
    first, v = [], 0
    while v < n:
        k = int(rng.integers(4, 8))
        if n - v - k < 4:
            k = n - v
        first.append(v)
        v += k
    first.append(n)
    e = []
    for g, (a, b) in enumerate(zip(first, first[1:])):
        e += [(i, i + 1 if i + 1 < b else a) for i in range(a, b)]
        for t in range(1 + links):
            h = g + 1 if t == 0 else int(rng.integers(g + 1, g + 40))
            if h < len(first) - 1:
                e.append((int(rng.integers(a, b)), int(rng.integers(first[h], first[h + 1]))))
    a, b = first[0], first[1]
    e += [(i, j) for i in range(a, b) for j in range(a, b) if i != j]
    ids = rng.permutation(n) if shuffle else np.arange(n)
    e = ids[np.asarray(e)]
    return O.build_csr(n, e[:, 0].astype(np.int32).copy(), e[:, 1].astype(np.int32).copy())


@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("links", [0, 6])
@pytest.mark.parametrize("n", [40, 1020, 1029, 1030, 1031, 1032, 1033, 1040, 5000, 70001])
def test_colouring_by_one_block_and_by_all(n, links, shuffle):
    g = cycles(n, links, n + links, shuffle)
    want = O.tarjan(g)
    with I.Solver(0) as s:
        for h in (g, O.Graph(g.bw_beg, g.bw_adj, g.fw_beg, g.fw_adj)):
            s.upload(I.HostGraph(h.fw_beg, h.fw_adj, h.bw_beg, h.bw_adj))
            s.solve(I.default_params(wcc_mode=2))
            assert np.array_equal(s.labels(), want)


@pytest.mark.parametrize("seed", [0, 1])
@pytest.mark.parametrize("n", [40, 700, 1040, 3001])
@pytest.mark.parametrize("more", [-1, 0])  # one edge short of 32 a vertex, and 32
def test_colouring_at_the_dense_line(n, more, seed):
    """Lists so long that a block sweeps once between grid barriers, and one
    edge short of that: cycles with extra edges forward (and back
    where the ids are too few for that)."""
    rng = np.random.default_rng(100 * n + seed)
    base = cycles(n, 2, n + seed, False)
    src = np.repeat(np.arange(n), np.diff(base.fw_beg))
    have = np.unique(src * n + base.fw_adj)
    room = np.setdiff1d(np.flatnonzero(np.triu(np.ones((n, n), bool), 1).ravel()), have)
    extra = rng.permutation(room)[:32 * n + more - have.size]
    if extra.size < 32 * n + more - have.size:  # 40 vertices: past the upper triangle too
        low = np.setdiff1d(np.flatnonzero(np.tril(np.ones((n, n), bool), -1).ravel()), have)
        extra = np.concatenate([extra, rng.permutation(low)[:32 * n + more - have.size - extra.size]])
    e = np.concatenate([have, extra])
    g = O.build_csr(n, (e // n).astype(np.int32), (e % n).astype(np.int32))
    assert g.fw_adj.size == 32 * n + more
    want = O.tarjan(g)
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        s.solve(I.default_params(wcc_mode=2))
        assert np.array_equal(s.labels(), want)
