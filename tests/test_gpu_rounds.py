"""The time-stepped rounds of -bfs against the oracle: sizes, radius, ids and keys of every level, and the labels.  By
default only levels of 2^20 vertices and more that are skewed, or whose deviates do not fit packed keys, run in rounds,
so the small graphs ask for them with the options that have every level run so (the default cut-over to sweeps given
outright, other cut-overs, pushes only, directions chosen on every level), and large graphs take the default.  Each
run's launches say which schedule it ran."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu

FORCED = [dict(tail_sweeps=3), dict(tail_sweeps=-1), dict(tail_sweeps=1), dict(pull_rounds=-1), dict(pull_rounds=1),
          dict(tail_sweeps=-1, pull_rounds=1)]


def graph(case):
    if case == "gnm":
        return ca.generate("gnm_undirected", n=1 << 14, m=1 << 15, seed=3)
    if case == "grid2":
        return ca.generate("grid_2d", nx=128, ny=100, p=0.55, seed=2)
    if case == "grid3":
        return ca.generate("grid_3d", nx=24, ny=24, nz=24, p=0.3, seed=2)
    if case == "rmat":
        return ca.generate("rmat", n=1 << 13, m=1 << 16, seed=3)
    if case == "path":
        return ca.Graph.from_edges(5000, [(i, i + 1) for i in range(4999)])
    if case == "star":
        return ca.Graph.from_edges(20001, [(0, i) for i in range(1, 20001)] + [(i, i + 1) for i in range(1, 1000)])
    assert case == "ordered"  # level 0 of 2^16 vertices and more: stored in degree order
    return ca.generate("rmat", n=1 << 17, m=1 << 20, seed=5)


def check(g, run, **kw):
    dg = ca.DeviceGraph(g)
    try:
        lab, st = dg.find_components(variant="exp", use_bfs=True, record_trace=True, **kw)
        tr = dg.trace()
    finally:
        dg.close()
    assert st["kernel_launches"]["round"] > 0, kw
    want = run.levels()
    assert len(tr) == len(want), kw
    for lvl, ((info, keys, gid), winfo) in enumerate(zip(tr, want)):
        assert (info[0], info[1], info[3]) == (winfo[0], winfo[1], winfo[3]), (kw, lvl)
        wkeys, wgid = run.level_keys(lvl)
        assert np.array_equal(gid, wgid), (kw, lvl)
        assert np.array_equal(keys, wkeys), (kw, lvl)
    assert np.array_equal(lab, run.labels()), kw
    return st


@pytest.mark.parametrize("stream", [ca.STREAM_REFERENCE, ca.STREAM_HASHED])
@pytest.mark.parametrize("case", ["gnm", "grid2", "grid3", "rmat", "path", "star", "ordered"])
def test_forced_rounds(case, stream):
    g = graph(case)
    okw = dict(seed=1005, seq_limit=64, stream=stream)
    run = oracle.Run(g.offsets, g.targets, variant="exp", keep_keys=True, **okw)
    for sched in FORCED:
        print(case, stream, sched, flush=True)
        check(g, run, **okw, **sched)
    if case == "ordered":
        check(g, run, **okw, tail_sweeps=3, input_order=True)


@pytest.mark.parametrize("stream", [ca.STREAM_REFERENCE, ca.STREAM_HASHED])
def test_forced_rounds_with_replicas(stream):
    for name, g, thr in (("star", ca.Graph.from_edges(3001, [(0, i) for i in range(1, 3001)]), 16.0),
                         ("rmat", graph("rmat"), 2.0)):
        okw = dict(seed=1007, seq_limit=64, stream=stream, replicate=True, hd_threshold=thr)
        run = oracle.Run(g.offsets, g.targets, variant="exp", keep_keys=True, **okw)
        for sched in FORCED[:2]:
            print(name, sched, flush=True)
            st = check(g, run, **okw, **sched)
            assert (st["hubs"], st["replicas"]) == run.replication()


@pytest.mark.parametrize("mode", ["local", "single", "double"])
def test_forced_rounds_after_pre_contraction(mode):
    g = ca.generate("gnm_undirected", n=1 << 14, m=1 << 15, seed=3)
    okw = dict(seed=1005, seq_limit=64, stream=ca.STREAM_HASHED, pre_contract=mode, pre_blocks=64)
    run = oracle.Run(g.offsets, g.targets, variant="exp", keep_keys=True, **okw)
    for sched in FORCED[:2]:
        check(g, run, **okw, **sched)


def test_default_rounds_on_a_large_skewed_level():
    g = ca.generate("rmat", n=1 << 21, m=1 << 24, seed=3)
    assert int((np.diff(g.offsets.astype(np.int64)) > 0).sum()) >= 1 << 20
    okw = dict(seed=5, seq_limit=1 << 14, stream=ca.STREAM_HASHED)
    run = oracle.Run(g.offsets, g.targets, variant="exp", keep_keys=True, **okw)
    check(g, run, **okw)
    check(g, run, **okw, tail_sweeps=-1)


@pytest.mark.parametrize("beta,rounds", [(0.1, False), (0.02, True)])
def test_default_schedule_by_rate(beta, rounds):
    g = ca.generate("gnm_undirected", n=1100000, m=2500000, seed=3)
    assert int((np.diff(g.offsets.astype(np.int64)) > 0).sum()) >= 1 << 20
    kw = dict(variant="exp", seed=5, seq_limit=1 << 14, stream=ca.STREAM_HASHED, beta=beta)
    run = oracle.Run(g.offsets, g.targets, **kw)
    lv = run.levels()
    lab, st = ca.find_components(g, use_bfs=True, **kw)
    assert np.array_equal(lab, run.labels())
    assert (st["levels"], st["radius_sum"]) == (len(lv), sum(x[3] for x in lv))
    assert (st["kernel_launches"]["round"] > 0) == rounds
