"""The one-workgroup tail of the contraction against the oracle: labels, levels and radii, which depend on the
graph and the deviates alone.  Graphs start at level 0 inside the tail or one vertex or edge slot outside
it (kTailSmall = 16128 and kTailVertices = 32768 vertices, 2^19 and 2^18 edge slots), cut-offs lie on both
sides of a level's exact number of edges (small ones and ones that need several hash parts), and the tail
starts below general levels too.  With record_trace the general path runs every level: the two agree."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu


def connected(rng, n, m):
    """n vertices without isolated ones, exactly m simple edges: a ring and random chords."""
    ring = np.stack([np.arange(n), (np.arange(n) + 1) % n], 1)
    ring = np.sort(ring, 1)
    have = np.unique(ring[:, 0] * n + ring[:, 1])
    more = rng.integers(0, n, size=(2 * (m - n) + 64, 2))
    more = np.sort(more[more[:, 0] != more[:, 1]], 1)
    keys = np.setdiff1d(np.unique(more[:, 0] * n + more[:, 1]), have)
    keys = np.concatenate([have, rng.permutation(keys)[: m - n]])
    assert len(keys) == m
    return ca.Graph.from_edges(n, np.stack([keys // n, keys % n], 1))


def check(g, **kw):
    okw = {k: v for k, v in kw.items() if k != "use_bfs"}
    run = oracle.Run(g.offsets, g.targets, **okw)
    lv = run.levels()
    dg = ca.DeviceGraph(g)
    lab, st = dg.find_components(**kw)
    lab2, st2 = dg.find_components(record_trace=True, **kw)
    dg.close()
    assert np.array_equal(lab, run.labels()) and np.array_equal(lab2, lab)
    want = (len(lv), sum(x[3] for x in lv))
    assert (st["levels"], st["radius_sum"]) == want, kw
    assert (st2["levels"], st2["radius_sum"]) == want, kw
    assert st["components"] == st2["components"]
    return lv


@pytest.mark.parametrize("n,m", [(2, 1), (3, 3), (700, 900), (16127, 20000), (16128, 20000), (16129, 20000), (16000, 262144),
                                 (16000, 262145), (32767, 40000), (32768, 40000), (32769, 40000), (20000, 131072),
                                 (20000, 131073)])
def test_sizes(n, m):
    rng = np.random.default_rng(n + m)
    g = connected(rng, n, m) if n > 3 else ca.Graph.from_edges(n, [(i, (i + 1) % n) for i in range(n)])
    print(f"tail n={g.n} m={g.m}", flush=True)
    check(g, variant="exp", seed=1003, seq_limit=64, stream=ca.STREAM_HASHED)
    check(g, variant="exp", seed=1003, seq_limit=0, stream=ca.STREAM_HASHED, use_bfs=True)
    check(g, variant="local", seed=1003, seq_limit=64)


@pytest.mark.parametrize("use_bfs", [False, True])
@pytest.mark.parametrize("stream", [ca.STREAM_HASHED, ca.STREAM_REFERENCE])
def test_cut_off_is_exact(stream, use_bfs):
    rng = np.random.default_rng(5)
    for g in (connected(rng, 6000, 30000), connected(rng, 9000, 120000)):
        lv = check(g, variant="exp", seed=7, seq_limit=1, stream=stream, use_bfs=use_bfs)
        for x in lv[:4]:
            for seq in (x[1] - 1, x[1], x[1] + 1):
                print(f"cut-off {seq} of level edges {[y[1] for y in lv]}", flush=True)
                check(g, variant="exp", seed=7, seq_limit=max(int(seq), 1), stream=stream, use_bfs=use_bfs)


def test_tail_below_general_levels():
    g = ca.generate("gnm_undirected", n=60000, m=200000, seed=3)
    for kw in (dict(variant="exp", stream=ca.STREAM_HASHED), dict(variant="exp", stream=ca.STREAM_REFERENCE),
               dict(variant="local")):
        lv = check(g, seed=11, seq_limit=100, **kw)
        assert len(lv) > 1 and lv[1][0] <= 16128  # levels 1 and on run in the tail
    check(ca.generate("grid_3d", nx=40, ny=40, nz=40, p=0.3, seed=3), variant="exp", seed=2, seq_limit=100,
          stream=ca.STREAM_HASHED, use_bfs=True)


def test_repeated_edges_and_hubs():
    # rows that list a neighbour several times; a hub; several components
    off = np.array([0, 3, 5, 8, 10, 11, 12, 13], np.uint64)
    tgt = np.array([1, 1, 2, 0, 2, 0, 1, 3, 2, 2, 5, 4, 3], np.uint32)
    g = ca.Graph(off[:7], tgt[:12])
    check(g, variant="exp", seed=3, seq_limit=0, stream=ca.STREAM_HASHED, use_bfs=True)
    star = ca.Graph.from_edges(12001, [(0, i) for i in range(1, 12001)] + [(i, i + 1) for i in range(1, 3000)])
    check(star, variant="exp", seed=4, seq_limit=16, stream=ca.STREAM_HASHED)
    check(star, variant="exp", seed=4, seq_limit=16, stream=ca.STREAM_HASHED, replicate=True, hd_threshold=4.0)


def test_level_cap_and_small_rates():
    rng = np.random.default_rng(8)
    g = connected(rng, 3000, 6000)
    dg = ca.DeviceGraph(g)
    with pytest.raises(ca.KcError) as e:
        dg.find_components(seed=3, seq_limit=0, stream=ca.STREAM_HASHED, max_levels=1)
    assert e.value.code == ca.KC_ERR_INVALID and "1 levels" in str(e.value)
    lab, _ = dg.find_components(seed=3, seq_limit=0, stream=ca.STREAM_HASHED)
    dg.close()
    assert np.array_equal(lab, oracle.canonical_labels(g.offsets, g.targets))
    # deviates above 2^17 - 3 do not fit the packed keys: the general path
    check(g, variant="exp", seed=3, seq_limit=64, stream=ca.STREAM_HASHED, beta=2e-4)
    check(g, variant="exp", seed=3, seq_limit=64, stream=ca.STREAM_HASHED, beta=4e-4)
