"""Adjacency entries read top-down, as the kernel profile gives them: with
every level top-down, each list of what is reached is read once, whether a grid,
a block or one wave read it."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O
from ispan_amd import hiprt as H
from tests.test_gpu_narrow_exits import repeated

pytestmark = pytest.mark.gpu


def beside_a_cycle(g, n):
    """g and a cycle of n vertices, which keeps so much unvisited that no
    traversal of g goes bottom-up."""
    src = np.repeat(np.arange(g.V), np.diff(g.fw_beg))
    c = np.arange(n)
    return O.build_csr(g.V + n, np.concatenate([src, g.V + c]).astype(np.int32),
                       np.concatenate([g.fw_adj, g.V + (c + 1) % n]).astype(np.int32))


@pytest.mark.parametrize("local", [64, 0])
@pytest.mark.parametrize("shape", [(2,), (3, 2, 2), (1, 600), (40, 70), (20, 20, 20)], ids=str)
def test_top_down_edges(shape, local):
    one = repeated(shape, 12, 300, False)
    g = beside_a_cycle(one, 200_000)
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        st = s.solve(I.default_params(alpha=1, td_local=local))
        assert np.array_equal(s.labels(), O.tarjan(g))
        kp = s.kernel_profile()
    assert st.fw_size == st.bw_reach == one.V
    assert kp.edges[2] == 0 and kp.found[2] == 0
    assert kp.edges[0] == 2 * one.fw_adj.size
    assert kp.found[0] == 2 * (one.V - 1)


def unreachable_lists(heavy, lists, leaves, path, V):
    """A pivot with `leaves` neighbours and a path from it, all edges both
    ways, and beside it `lists` vertices B joined both ways to all of `heavy`:
    active, and not reached, so that every bottom-up level reads their lists
    to the end."""
    rng = np.random.default_rng(1)
    free = np.setdiff1d(rng.permutation(V)[:lists + leaves + path + len(heavy) + 1], heavy)
    rng.shuffle(free)
    B, free = free[:lists], free[lists:]
    hub, free = free[0], free[1:]
    leaf, p = free[:leaves], np.concatenate([[hub], free[leaves:leaves + path]])
    src = np.concatenate([np.repeat(heavy, lists), np.full(leaves, hub), p[:-1]]).astype(np.int32)
    dst = np.concatenate([np.tile(B, len(heavy)), leaf, p[1:]]).astype(np.int32)
    return np.concatenate([src, dst]), np.concatenate([dst, src]), hub


@pytest.mark.parametrize("runs,lists,path", [([0], 6000, 1), ("one block's", 6000, 200)], ids=["wave", "block"])
def test_bottom_up_edges(runs, lists, path):
    """Entries read bottom-up: more than 2^20 by one wave, and more than 2^32
    by one block over the levels of a traversal."""
    V = 1 << 20
    if runs == "one block's":
        # the runs of 512 vertices of block 0's waves, where both directions
        # are bottom-up: 2048 waves a direction on 256 CUs
        total = 256 * 16
        m = 2654435761 % total
        while np.gcd(m, total) != 1:
            m += 1
        runs = [w * m % 2048 for w in range(8)]
    heavy = np.concatenate([np.arange(512) + 512 * r for r in runs])
    src, dst, hub = unreachable_lists(heavy, lists, 7000, path, V)
    beside = 2 * lists * heavy.size
    a, b = H.DeviceArray(src), H.DeviceArray(dst)
    with I.Solver(0) as s:
        dg = s.build_csr(V, src.size, a.ptr, b.ptr)
        a.free()
        b.free()
        try:
            s.bind(dg)
            big = 2**31 - 1
            st = s.solve(I.default_params(alpha=big, beta=big, gamma=big))
            kp = s.kernel_profile()
        finally:
            dg.free()
    assert (st.pivot, st.fw_size, st.bw_reach) == (hub, 7001 + path, 7001 + path)
    levels = (st.fw_levels - 1) + (st.bw_levels - 1)  # all but level 0 bottom-up
    if path == 1:
        assert levels == 2 and kp.edges[2] == 2 * beside
    else:
        assert levels * beside // 2 > 1 << 32  # the heavy vertices' half of the lists
        # and at most the path's own entries
        assert levels * beside <= kp.edges[2] <= levels * (beside + 2 * path)
    assert kp.edges[0] == 2 * (7000 + 1)
