"""Sweeps that do not read settled rows again, and the schedules a level may run in, against the oracle: labels,
levels and radii.  Long paths (distances far above the number of sweeps), hubs cut into chunks, keys that do not
fit the packed form (a small beta), levels below and above the packed keys' 2^16 vertices, a skewed graph of more
than 2^20 vertices (rounds)."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu

SCHEDULES = [dict(), dict(use_bfs=True), dict(use_bfs=True, tail_sweeps=-1), dict(use_bfs=True, tail_sweeps=1),
             dict(use_bfs=True, pull_rounds=1)]


def graphs():
    rng = np.random.default_rng(1)
    v = np.arange(70000)
    perm = rng.permutation(70000)
    yield "path", ca.Graph.from_edges(70000, np.stack([perm[:-1], perm[1:]], 1))
    hub = np.stack([np.zeros(69999, np.int64), v[1:]], 1)[::2]
    yield "caterpillar", ca.Graph.from_edges(70000, np.concatenate([hub, np.stack([v[1:-1], v[2:]], 1)]))
    yield "small", ca.generate("gnm_undirected", n=40000, m=50000, seed=4)
    yield "grid", ca.generate("grid_2d", nx=500, ny=300, p=0.6, seed=4)
    yield "rmat", ca.generate("rmat", n=1 << 17, m=1 << 20, seed=4)


@pytest.mark.parametrize("beta", [0.1, 0.02])
def test_schedules(beta):
    for name, g in graphs():
        for stream in (ca.STREAM_HASHED, ca.STREAM_REFERENCE):
            kw = dict(variant="exp", seed=3, seq_limit=16, stream=stream, beta=beta)
            run = oracle.Run(g.offsets, g.targets, **kw)
            lv = run.levels()
            dg = ca.DeviceGraph(g)
            for sched in SCHEDULES:
                print(name, beta, stream, sched, flush=True)
                lab, st = dg.find_components(**kw, **sched)
                assert np.array_equal(lab, run.labels())
                assert (st["levels"], st["radius_sum"]) == (len(lv), sum(x[3] for x in lv)), (name, sched)
            dg.close()


def test_large_skewed_level():
    g = ca.DeviceGraph.generate("rmat", n=1 << 22, m=1 << 24, seed=6)
    kw = dict(variant="exp", seed=3, seq_limit=1 << 16, stream=ca.STREAM_HASHED)
    ref, want = g.find_components(**kw)
    for sched in SCHEDULES[1:]:
        lab, st = g.find_components(**kw, **sched)
        assert np.array_equal(lab, ref)
        assert (st["levels"], st["radius_sum"], st["components"]) == (want["levels"], want["radius_sum"], want["components"])
    g.close()
