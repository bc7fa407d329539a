"""The bin autotuner on calls that use no bins (every level in one workgroup; shortcuts): the thresholds' times are the
same launches' noise there, so the defaults stay.  On a graph whose levels do use them a choice is a timed candidate."""
import pytest

import components_amd as ca

pytestmark = pytest.mark.gpu

DEFAULTS = (16, 256, 4096)


def test_unused_bins_keep_the_defaults():
    small = [ca.generate("gnm_undirected", n=n, m=2 * n, seed=n) for n in (50, 1000, 3000, 12000)]
    calls = [(g, dict(seed=3, stream=ca.STREAM_HASHED)) for g in small]
    calls += [(ca.generate("grid_2d", nx=300, ny=200, p=0.6, seed=s), dict(seed=3, variant="shortcut")) for s in (1, 2)]
    for g, kw in calls:
        dg = ca.DeviceGraph(g)
        for _ in range(3):
            t = dg.autotune(**kw)
            print(g.n, kw, t, flush=True)
            assert (t["small"], t["mid"], t["large"]) == DEFAULTS and t["ms"] == t["default_ms"]
        dg.close()


def test_used_bins_are_chosen_by_time():
    g = ca.generate("rmat", n=1 << 17, m=1 << 20, seed=5)
    dg = ca.DeviceGraph(g)
    t = dg.autotune(seed=3, stream=ca.STREAM_HASHED)
    dg.close()
    assert t["candidates"] == 27
    if (t["small"], t["mid"], t["large"]) != DEFAULTS:
        assert t["ms"] <= 0.98 * t["default_ms"]
