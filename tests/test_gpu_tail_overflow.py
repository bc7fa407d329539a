"""The tail's count of a level's edges where one hash part outgrows its table, and the start over on the general path
that follows.  The parts are cut by the edges' hash, so it takes a graph made for it: most vertices draw the distance 0
and keep their own cluster, the others hang on vertex 0 and join its cluster, so the second level's indices are known,
and only edges whose second-level pair falls into the same part are taken."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu

TABLE, LOAD = 1 << 15, 20000  # slots of a part's table, edges a part is meant to hold


def edge_hash(x):
    x = x.astype(np.uint32)
    x = (x ^ (x >> 15)) * np.uint32(0x2c1b3c6d)
    x = (x ^ (x >> 12)) * np.uint32(0x297a2d39)
    return x ^ (x >> 15)


def crowded_graph(n, total, seed, beta):
    """A graph of `total` vertices, the first n with edges, whose second level has 39000 edges or a few more, all in the
    second of two parts."""
    dev = np.array([oracle.hashed_deviate(v, seed, 1, beta) for v in range(n)])
    centres = np.flatnonzero(dev == 0)  # the second level's vertices, in its order
    assert dev[0] == 0
    rng = np.random.default_rng(1)

    def upper_half(a, b):
        lo, hi = np.minimum(a, b), np.maximum(a, b)
        return (lo != hi) & (edge_hash(lo | hi << 16) >> 31 == 1)

    k = len(centres)
    a, b = rng.integers(0, k, 200000), rng.integers(0, k, 200000)
    ok = upper_half(a, b)
    a, b = a[ok][:39000], b[ok][:39000]
    left = np.setdiff1d(np.arange(k), np.concatenate([a, b]))  # every centre has an edge
    partner = [next(w for w in range(k) if upper_half(np.array([v]), np.array([w]))[0]) for v in left]
    a, b = np.concatenate([a, left]), np.concatenate([b, np.array(partner, np.int64)])
    lo, hi = np.minimum(a, b), np.maximum(a, b)
    pairs = np.unique(lo * n + hi)
    assert TABLE < len(pairs) <= 2 * LOAD
    edges = np.stack([centres[pairs // n], centres[pairs % n]], 1)
    others = np.flatnonzero(dev)
    return ca.Graph.from_edges(total, np.concatenate([edges, np.stack([np.zeros_like(others), others], 1)])), len(pairs)


@pytest.mark.parametrize("total", [16000, 70000])  # the labels of the second go through helper threads
def test_full_part_starts_over(total):
    seed, beta = 3, 5.0
    g, edges = crowded_graph(16000, total, seed, beta)
    kw = dict(variant="exp", seed=seed, beta=beta, stream=ca.STREAM_HASHED, seq_limit=edges - 50)
    run = oracle.Run(g.offsets, g.targets, **kw)
    lv = run.levels()
    print(f"levels {lv}", flush=True)
    assert lv[1][1] == edges and len(lv) >= 2
    dg = ca.DeviceGraph(g)
    for _ in range(2):
        lab, st = dg.find_components(**kw)
        # the general path ran, although the graph fits the tail
        assert st["kernel_launches"]["relabel"] > 0
        assert np.array_equal(lab, run.labels())
        assert (st["levels"], st["radius_sum"]) == (len(lv), sum(x[3] for x in lv))
    # the same graph with a cut-off that one table holds stays in the tail
    lab, st = dg.find_components(**dict(kw, seq_limit=64, beta=0.1))
    dg.close()
    assert st["kernel_launches"]["relabel"] == 0
    assert np.array_equal(lab, oracle.canonical_labels(g.offsets, g.targets))
