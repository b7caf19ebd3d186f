"""The level trace (ISPAN_LEVEL_TRACE): every level of either direction has its
blocks' times, also where both directions are bottom-up side by side."""
import re

import pytest

import ispan_amd as I

pytestmark = pytest.mark.gpu

LINE = re.compile(r"(FW|BW) level +(\d+) (TD|BU) found +(\d+) edges +(-?\d+) +([\d.-]+) ms +work ([\d.-]+)\.\.([\d.-]+) "
                  r"max block scan (\d+) marks dense ([\d.-]+) probed ([\d.-]+) misses ([\d.-]+)")


@pytest.mark.parametrize("kind", ["rmat", "grid"])
def test_every_level_has_its_times(kind, monkeypatch, capfd):
    monkeypatch.setenv("ISPAN_LEVEL_TRACE", "1")
    with I.Solver(0) as s:
        g = s.gen_rmat(1 << 20, 16.0, 1) if kind == "rmat" else s.gen_grid(300, 0.6, 1)
        s.bind(g)
        s.solve()
        capfd.readouterr()
        st = s.solve()
        kp = s.kernel_profile()
        text = capfd.readouterr().err
        g.free()
    levels = [m.groups() for m in map(LINE.search, text.splitlines()) if m]
    for name, n in (("FW", st.fw_levels), ("BW", st.bw_levels)):
        assert [int(x[1]) for x in levels if x[0] == name] == list(range(n))
    side = {x[1] for x in levels if x[:1] == ("FW",) and x[2] == "BU"} & {x[1] for x in levels if x[0] == "BW" and x[2] == "BU"}
    assert side or kind == "grid"
    for d, lv, mode, found, edges, ms, lo, hi, scan, dense, probed, misses in levels:
        assert 0 <= float(lo) <= float(hi) <= float(ms) + 0.01, (d, lv)
        if mode == "BU":
            assert float(hi) > 0 and 0 < float(probed) <= float(misses) <= float(hi) + 0.001, (d, lv)
    assert sum(int(x[4]) for x in levels if x[2] == "TD") == kp.edges[0]
    assert sum(int(x[4]) for x in levels if x[2] == "BU") == kp.edges[2]
    assert sum(int(x[3]) for x in levels) == kp.found[0] + kp.found[2]
