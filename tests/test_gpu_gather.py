"""Traversals that come back from bottom-up with much left to claim: whatever
is found or claimed is queued once, so its list is read once, also where waves
claim while others still gather (more than one group of words a wave beyond
2^24 vertices)."""
import numpy as np
import pytest

import ispan_amd as I
from ispan_amd import hiprt as H

pytestmark = pytest.mark.gpu


def wide(V, deg, hub, seed):
    """Strongly connected: a cycle through all V vertices in random order,
    `deg` random edges each, and vertex 7 with `hub` out- and in-edges, which
    makes it the pivot.  Its list has more than one piece (256 edges), so that
    level 0 stays one level."""
    rng = np.random.default_rng(seed)
    p = rng.permutation(V).astype(np.int32)
    src = [p] + [np.arange(V, dtype=np.int32)] * deg
    dst = [np.roll(p, -1)] + [rng.integers(0, V, V).astype(np.int32) for _ in range(deg)]
    h = rng.integers(0, V, (2, hub)).astype(np.int32)
    src += [np.full(hub, 7, np.int32), h[0]]
    dst += [h[1], np.full(hub, 7, np.int32)]
    return np.concatenate(src), np.concatenate(dst)


@pytest.mark.parametrize("V,deg,hub", [(3000, 1, 600), (70_001, 2, 600), (400_000, 0, 3000), (2_000_003, 2, 50_000),
                                       ((1 << 24) + 70_000, 2, 200_000), ((1 << 25) + 5, 0, 2000)])
def test_lists_are_read_once_after_the_gather(V, deg, hub):
    src, dst = wide(V, deg, hub, V % 1000)
    a, b = H.DeviceArray(src), H.DeviceArray(dst)
    with I.Solver(0) as s:
        dg = s.build_csr(V, src.size, a.ptr, b.ptr)
        a.free()
        b.free()
        try:
            g = dg.download()
            s.bind(dg)
            seen = {}
            for local in (64, 1, 0):
                # bottom-up from level 1 on, for one level
                st = s.solve(I.default_params(alpha=2**31 - 1, gamma=0, td_local=local))
                kp = s.kernel_profile()
                assert (st.pivot, st.fw_size, st.bw_reach, st.giant_size) == (7, V, V, V)
                assert not s.labels().any()
                # all lists but those of the pivot's neighbours, claimed at
                # level 0: no later level goes back to them
                want = 0
                for beg, adj in ((g.fw_beg, g.fw_adj), (g.bw_beg, g.bw_adj)):
                    first = adj[beg[7]:beg[8]]
                    want += int(dg.E) - int((beg[first + 1] - beg[first]).sum())
                assert kp.edges[0] == want, local
                assert kp.found[0] + kp.found[2] == 2 * (V - 1)
                seen[local] = kp.found[2]
            assert min(seen.values()) < 2 * (V - 1)  # and there was something left
            # the sums over the forward set and the giant come from the bitmaps
            s.solve_stats(st)
            assert (st.fw_edges, st.bw_edges, st.n_scc) == (dg.E, dg.E, 1)
        finally:
            dg.free()


@pytest.mark.parametrize("gamma", [0, 1, 3])
@pytest.mark.parametrize("kind", ["rmat", "sparse", "grid"])
def test_labels_and_reach_after_the_gather(kind, gamma):
    """Against the engine that goes level by level from the host."""
    with I.Solver(0) as s:
        dg = s.gen_grid(1500, 0.6, 3) if kind == "grid" else \
            s.gen_rmat(1_500_001, 3.0 if kind == "sparse" else 12.0, 5)
        try:
            s.bind(dg)
            ref = s.solve_stats(s.solve(I.default_params(engine=1)))
            want = s.labels()
            for alpha in (30, 2**31 - 1):
                for local in (64, 1, 0):
                    st = s.solve(I.default_params(alpha=alpha, gamma=gamma, td_local=local))
                    assert np.array_equal(s.labels(), want)
                    s.solve_stats(st)
                    for k in ("fw_size", "giant_size", "fw_edges", "bw_edges", "n_scc"):
                        assert getattr(st, k) == getattr(ref, k), k
        finally:
            dg.free()
