"""Small WCCs after the trims: sizes around the 1-, 2- and 4-word closure
rows and past them, dense and path-like, long lists, shuffled ids, on both
engines, against Tarjan."""
import numpy as np
import pytest

import ispan_amd as I
import oracle as O

pytestmark = pytest.mark.gpu


def wccs(sizes, seed, shape):
    """Disjoint WCCs of the given sizes, ids shuffled.  chain: cycles of 2 to
    5 vertices, each with edges to the next two; ring: one cycle; dense: random
    edges (several SCCs, long lists when large)."""
    rng = np.random.default_rng(seed)
    e, v = [], 0
    for n in sizes:
        if shape == "ring":
            e += [(v + i, v + (i + 1) % n) for i in range(n)]
        elif shape == "dense":
            e += [(v + i, v + i + 1) for i in range(n - 1)]
            a = rng.integers(0, n, (2, 3 * n + (200 if n > 64 else 0)))
            a[0, :100 if n > 64 else 0] = 0  # a list of more than a wave
            back = rng.random(a.shape[1]) < 0.3
            lo, hi = np.minimum(a[0], a[1]), np.maximum(a[0], a[1])
            e += list(zip(v + np.where(back, hi, lo), v + np.where(back, lo, hi)))
        else:
            b, starts = 0, []
            while b < n:
                k = min(int(rng.integers(2, 6)), n - b)
                starts.append(b)
                e += [(v + b + i, v + b + (i + 1) % k) for i in range(k)]
                b += k
            e += [(v + s + 0, v + t) for i, s in enumerate(starts) for t in starts[i + 1:i + 3]]
        v += n
    # a giant of its own, so that the rest is left to the mice phase
    e += [(v + i, v + (i + 1) % 50) for i in range(50)] + [(v, v + i) for i in range(2, 50)] + \
         [(v + i, v) for i in range(2, 50)]
    v += 50
    e = rng.permutation(v)[np.asarray(e, np.int64)]
    return O.build_csr(v, e[:, 0].astype(np.int32).copy(), e[:, 1].astype(np.int32).copy())


@pytest.mark.parametrize("shape", ["chain", "ring", "dense"])
@pytest.mark.parametrize("sizes", [
    list(range(4, 40)), [63, 64, 65], [127, 128, 129], [191, 192, 193, 255, 256], [257, 300, 1024], [1025, 7],
    [5] * 3000 + [200] * 20,
], ids=lambda s: f"{len(s)}to{max(s)}")
def test_small_wccs(sizes, shape):
    g = wccs(sizes, len(sizes), shape)
    want = O.tarjan(g)
    with I.Solver(0) as s:
        s.upload(I.HostGraph(g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj))
        for kw in ({}, {"wcc_mode": 1}, {"engine": 1}, {"trim_times": 0}):
            for _ in range(2):
                st = s.solve(I.default_params(**kw))
                assert np.array_equal(s.labels(), want), kw
        assert st.n_wcc <= len(sizes) and st.max_wcc <= max(sizes)
