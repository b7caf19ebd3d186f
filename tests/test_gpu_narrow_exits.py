"""A narrow frontier that leaves its block again and again within one
traversal, for each reason it can leave: more edges than a block's step, a hub,
more entries than a tile holds, entries that had to be flushed.  All waves of
the block have to leave together, with what each of them holds."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O

pytestmark = pytest.mark.gpu

# a vertex's children, their children each, ..
SHAPES = {
    "edges": (300, 10),      # 3000 edges in 300 entries
    "edges just": (32, 64),  # 2048, which stay, and their 2048 back
    "edges past": (32, 65),  # 2080
    "hub": (1, 600),
    "hub among others": (40, 1),
    "entries": (1100,),
    "flushed": (1000, 3, 1),
}


def repeated(shape, times, path, hub):
    """`times` trees of the shape on a cycle, `path` vertices between them;
    every leaf has an edge to the next path.  hub: one child has 700 more
    leaves."""
    src, dst = [], []
    v = 0  # the path's last vertex so far
    for t in range(times):
        level = np.arange(v, v + 1)
        n = v + 1
        leaves = []
        for k, width in enumerate(shape):
            kids = n + np.arange(level.size * width)
            src.append(np.repeat(level, width))
            dst.append(kids)
            n += kids.size
            if hub and k == 0:
                more = n + np.arange(700)
                src.append(np.full(700, kids[kids.size // 2]))
                dst.append(more)
                leaves.append(more)
                n += 700
            level = kids
        leaves.append(level)
        ends = np.concatenate(leaves)
        src.append(ends)
        dst.append(np.full(ends.size, n))
        src.append(np.arange(n, n + path))
        dst.append(np.arange(n + 1, n + path + 1))
        v = n + path
    src.append(np.asarray([v]))
    dst.append(np.asarray([0]))
    p = np.random.default_rng(times).permutation(v + 1)
    return O.build_csr(v + 1, p[np.concatenate(src)].astype(np.int32), p[np.concatenate(dst)].astype(np.int32))


@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_every_exit_many_times(shape, flip):
    g = repeated(SHAPES[shape], 60, 7, shape == "hub among others")
    if flip:
        g = O.Graph(g.bw_beg, g.bw_adj, g.fw_beg, g.fw_adj)
    want = O.tarjan(g)
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        for alpha in (30, 1):  # bottom-up near the end, or hardly ever
            for _ in range(3):
                st = s.solve(I.default_params(alpha=alpha))
                assert np.array_equal(s.labels(), want)
                assert (st.fw_size, st.bw_reach, st.giant_size) == (g.V, g.V, g.V)
