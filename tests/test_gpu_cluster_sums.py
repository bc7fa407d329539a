"""Clusters placed by their running sums, against the oracle (labels, levels and radii): level sizes around the
workgroups' 4096 vertices and the scans' tiles of 2048 (runs of 512 a wave), one cluster holding nearly all of a level or thousands of small ones, buckets of every
dedup class, and levels on both sides of the dense cluster ids' bounds (2^20 vertices, average degree 8)."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu


def check(g, trace=True, **kw):
    """The trace keeps every level out of the one-workgroup tail."""
    okw = {k: v for k, v in kw.items() if k not in ("use_bfs", "input_order")}
    run = oracle.Run(g.offsets, g.targets, **okw)
    lv = run.levels()
    dg = ca.DeviceGraph(g)
    lab, st = dg.find_components(record_trace=trace, **kw)
    dg.close()
    assert np.array_equal(lab, run.labels())
    assert (st["levels"], st["radius_sum"]) == (len(lv), sum(x[3] for x in lv))
    return lv


@pytest.mark.parametrize("n", [2, 63, 511, 513, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 12289])
@pytest.mark.parametrize("shape", ["path", "star", "random", "cliques"])
def test_level_sizes(n, shape):
    rng = np.random.default_rng(n)
    v = np.arange(n)
    if shape == "path":
        e = np.stack([v[:-1], v[1:]], 1)
    elif shape == "star":  # one cluster takes nearly all; stars of its leaves keep cluster edges
        e = np.concatenate([np.stack([np.zeros(n - 1, np.int64), v[1:]], 1), np.stack([v[1:-1], v[2:]], 1)[::3]])
    elif shape == "random":
        e = rng.integers(0, n, size=(3 * n, 2))
        e = np.concatenate([e[e[:, 0] != e[:, 1]], np.stack([v, (v + 1) % n], 1)])
    else:
        e = np.concatenate([np.stack([v[v % 8 != 0] // 8 * 8, v[v % 8 != 0]], 1), np.stack([v[:-9:8], v[9::8]], 1)
                            if n > 64 else np.zeros((0, 2), np.int64)])
    e = np.unique(np.sort(e, 1), axis=0)
    g = ca.Graph.from_edges(n, e[e[:, 0] != e[:, 1]])
    print(f"sums {shape} n={n} m={g.m}", flush=True)
    check(g, variant="exp", seed=5, seq_limit=0, stream=ca.STREAM_HASHED, use_bfs=True)
    check(g, variant="exp", seed=6, seq_limit=0, stream=ca.STREAM_HASHED)
    check(g, variant="local", seed=5, seq_limit=0)


def test_bucket_classes():
    """A hub pair of 40000 leaves each and chords between them: small, medium and huge buckets in one level."""
    rng = np.random.default_rng(3)
    n = 120000
    leaf = np.arange(2, 80002)
    e = [np.stack([np.where(leaf % 2, 0, 1), leaf], 1)]
    e.append(rng.integers(2, n, size=(300000, 2)))
    e.append(np.stack([np.arange(80002, n - 1), np.arange(80003, n)], 1))
    e = np.sort(np.concatenate(e), 1)
    g = ca.Graph.from_edges(n, np.unique(e[e[:, 0] != e[:, 1]], axis=0))
    for kw in (dict(use_bfs=True), dict(), dict(input_order=True, use_bfs=True)):
        for trace in (True, False):
            check(g, trace=trace, variant="exp", seed=9, seq_limit=0, stream=ca.STREAM_HASHED, **kw)


@pytest.mark.parametrize("n,m", [((1 << 20) + 4096, 4 * (1 << 20) - 100000), ((1 << 20) + 4096, 4 * (1 << 20) + 200000),
                                 ((1 << 20) - 1, 5 << 20)])
def test_dense_id_bounds(n, m):
    """G(n, m) with nearly no isolated vertex: the average degree lies below or above 8, n below or above 2^20."""
    g = ca.generate("gnm_undirected", n=n, m=m, seed=2)
    check(g, trace=False, variant="exp", seed=4, seq_limit=4096, stream=ca.STREAM_HASHED, use_bfs=True, input_order=True)


@pytest.mark.parametrize("n", [1024 * 2048, 1024 * 2048 + 1])
def test_scan_levels(n):
    """A ring: the label scan takes two launches up to 1024 tiles, four above."""
    v = np.arange(n)
    g = ca.Graph.from_edges(n, np.stack([v, (v + 1) % n], 1))
    check(g, trace=False, variant="exp", seed=8, seq_limit=4096, stream=ca.STREAM_HASHED, use_bfs=True)
