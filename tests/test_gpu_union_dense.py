"""Union-find's rounds of hooks by size and density: below and at 2^14 vertices (edges sampled from every row), above 16
slots a vertex (an eighth of the shares), elsewhere two or three full rounds (2^19 vertices).  Labels of the shortcuts
variant, of the base case over the whole graph and of the pre-contraction's blocks, against the oracle.  Dense random
graphs, whose trees' links waited for one another, take no longer than sparser ones."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu


def check(g):
    ref = oracle.canonical_labels(g.offsets, g.targets)
    dg = ca.DeviceGraph(g)
    for kw in (dict(variant="shortcut"), dict(variant="exp", seq_limit=1 << 40)):
        for _ in range(2):
            lab, st = dg.find_components(**kw)
            assert np.array_equal(lab, ref), (g.n, g.m, kw)
            assert st["components"] == len(np.unique(ref))
    dg.close()


@pytest.mark.parametrize("n", [2, 37, (1 << 14) - 1, 1 << 14, (1 << 14) + 1, 70001])
@pytest.mark.parametrize("degree", [0.4, 1, 3, 15.5, 16.5, 60])
def test_random_graphs(n, degree):
    rng = np.random.default_rng(n)
    check(ca.Graph.from_edges(n, rng.integers(0, n, size=(max(1, int(n * degree / 2)), 2))))


def test_full_rounds_on_both_sides_of_their_bound():
    for n in ((1 << 19) - 1, 1 << 19):
        check(ca.generate("gnm_undirected", n=n, m=n, seed=2))
        check(ca.generate("gnm_undirected", n=n, m=9 * n, seed=2))


def test_dense_graphs_of_many_components():
    # cliques of 40, ids shuffled: dense, yet a tree each stays; and a hub beside them
    rng = np.random.default_rng(3)
    for cliques in (300, 700):
        i, j = np.triu_indices(40, 1)
        base = np.repeat(np.arange(cliques) * 40, len(i))
        e = np.stack([np.tile(i, cliques) + base, np.tile(j, cliques) + base], 1)
        n = 40 * cliques + 5000
        hub = np.stack([np.full(4999, 40 * cliques), np.arange(40 * cliques + 1, n)], 1)
        check(ca.Graph.from_edges(n, rng.permutation(n)[np.concatenate([e, hub])]))


def test_two_large_trees():
    # stars around the lowest ids (so that every leaf starts in its hub's tree) and many edges between their leaves,
    # which all find the same two roots; as many again in a third tree of its own
    rng = np.random.default_rng(8)
    n = 60000
    hub = rng.integers(0, 2, n)
    leaves = np.arange(3, n)
    stars = np.stack([hub[3:], leaves], 1)
    a, b = leaves[hub[3:] == 0], leaves[hub[3:] == 1]
    for cross in (1, 500, 400000):
        between = np.stack([rng.choice(a, cross), rng.choice(b, cross)], 1)
        check(ca.Graph.from_edges(n, np.concatenate([stars, between])))
        alone = np.stack([np.full(1000, n), n + 1 + np.arange(1000)], 1)
        check(ca.Graph.from_edges(n + 1001, np.concatenate([stars, alone, between])))


@pytest.mark.parametrize("blocks", [3, 64])
def test_blocks(blocks):
    for n, m in ((9000, 200000), (40000, 500000)):
        g = ca.generate("gnm_undirected", n=n, m=m, seed=5)
        kw = dict(seed=7, seq_limit=64, stream=ca.STREAM_HASHED, pre_contract="single", pre_blocks=blocks)
        run = oracle.Run(g.offsets, g.targets, variant="exp", **kw)
        lab, st = ca.find_components(g, **kw)
        assert np.array_equal(lab, run.labels())
        assert (st["levels"], st["radius_sum"]) == (len(run.levels()), sum(x[3] for x in run.levels()))


def test_dense_graphs_are_not_slower_than_sparse_ones():
    ms = []
    for degree in (8, 20, 40):
        dg = ca.DeviceGraph.generate("gnm_undirected", n=60000, m=60000 * degree // 2, seed=1)
        t = sorted(dg.find_components(variant="shortcut", copy_labels=False)[1]["time_ms"] for _ in range(21))
        ms.append(t[10])
        dg.close()
    print(f"8, 20 and 40 slots a vertex: {ms}", flush=True)
    assert max(ms[1:]) < 2 * ms[0]
