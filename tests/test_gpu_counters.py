"""Adjacency entries read top-down, as the kernel profile gives them: with
every level top-down, each list of what is reached is read once, whether a grid,
a block or one wave read it."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O
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
