"""The colouring method on a rest of more vertices than the line from which a
block sweeps once between grid barriers, and just below it, on lists whose
entries leave the active set round by round."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O
from ispan_amd import hiprt as H

pytestmark = pytest.mark.gpu

LINE = 2 * 256 * 1024  # two vertices for each of 256 blocks' threads


def quads(n, k, span, seed):
    """Cycles of four consecutive ids, and k edges a vertex forward to one of
    the next `span` ids."""
    rng = np.random.default_rng(seed)
    q = np.arange(n // 4 * 4)
    a = rng.integers(0, n, n * k)
    b = np.minimum(a + rng.integers(1, span, n * k), n - 1)
    return np.concatenate([q, a]).astype(np.int32), np.concatenate([q // 4 * 4 + (q + 1) % 4, b]).astype(np.int32)


@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("n,k,span", [(LINE, 1, 1 << 19), (LINE + 4, 1, 1 << 19), (LINE + 8, 1, 1 << 19),
                                      (LINE + 100_000, 5, 1 << 18), (LINE + 300_000, 1, 100_000)])
def test_wide_rest(n, k, span, flip):
    src, dst = quads(n, k, span, n + k)
    if flip:
        src, dst = dst, src
    a, b = H.DeviceArray(src), H.DeviceArray(dst)
    with I.Solver(0) as s:
        dg = s.build_csr(n, src.size, a.ptr, b.ptr)
        a.free()
        b.free()
        try:
            g = dg.download()
            s.bind(dg)
            st = s.solve(I.default_params(wcc_mode=2))
            got = s.labels()
        finally:
            dg.free()
    assert np.array_equal(got, O.tarjan(O.Graph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj)))
    assert st.giant_size == 4
