"""The batched form's LDS kernel at the edges of its size classes (1024 vertices and 4096 edges, 2048 and
12288, 4096 and 30592, 8192 and any): graphs with exactly as many vertices or edges as a class holds, one fewer and
one more (the last go to the next class or to the general kernel), rows on both sides of the 64
entries one thread reads, empty graphs and isolated vertices, and repeated edges, self-loops and
multiplicities that differ between the two directions.  Labels, levels and radii are compared with the
oracle on each graph alone, as in test_gpu_batch."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu

CLASSES = [(1024, 4096), (2048, 12288), (4096, 30592), (8192, 40000)]


def exact_graph(rng, n, m):
    """A simple graph with exactly m edges."""
    keys = np.unique(rng.integers(0, n * n, size=4 * m + 64))
    u, v = keys // n, keys % n
    keys = np.unique(np.minimum(u, v)[u != v] * n + np.maximum(u, v)[u != v])
    assert len(keys) >= m
    keys = rng.permutation(keys)[:m]
    return ca.Graph.from_edges(n, np.stack([keys // n, keys % n], 1))


def rows(n, lists):
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum([len(x) for x in lists])
    return ca.Graph(off, np.concatenate([np.asarray(x, np.uint32) for x in lists]).astype(np.uint32))


def check(graphs, seed, stream, beta=0.1, **tuning):
    b = ca.BatchGraphs.pack(graphs)
    db = ca.DeviceBatch(b)
    try:
        if tuning:
            db.set_tuning(**tuning)
        for rep in range(2):
            lab, st = db.run(seed=seed, stream=stream, beta=beta)
            levels, _, radius = db.graph_stats()
            for k, g in enumerate(graphs):
                run = oracle.Run(g.offsets, g.targets, variant="exp", seed=seed, seq_limit=0, stream=stream, beta=beta)
                lv = run.levels()
                a, z = int(b.vtx_off[k]), int(b.vtx_off[k + 1])
                assert np.array_equal(lab[a:z], run.labels()), (k, g.n, g.m)
                assert levels[k] == len(lv) and radius[k] == sum(x[3] for x in lv), (k, g.n, g.m)
    finally:
        db.close()


@pytest.mark.parametrize("cls", range(4))
def test_class_edges(cls):
    n, m = CLASSES[cls]
    rng = np.random.default_rng(cls)
    graphs = [exact_graph(rng, nn, mm) for nn in (n - 1, n, n + 1) for mm in (nn // 2, m // 2, m - 1, m, m + 1)]
    print(f"class {cls}: {[(g.n, g.m) for g in graphs]}", flush=True)
    check(graphs, 1001, ca.STREAM_HASHED, block=256, groups_per_cu=4, use_graph=bool(cls & 1))


def test_small_and_odd_graphs():
    rng = np.random.default_rng(9)
    none = ca.Graph(np.zeros(1, np.uint64), np.zeros(0, np.uint32))
    graphs = [none, ca.Graph(np.zeros(4, np.uint64), np.zeros(0, np.uint32)),
              ca.Graph.from_edges(3, [(0, 2)]),
              ca.Graph.from_edges(700, [(3, i) for i in range(4, 4 + 64)]),
              ca.Graph.from_edges(700, [(3, i) for i in range(4, 4 + 65)]),
              ca.Graph.from_edges(4096, [(4095, i) for i in range(4095)] + [(0, i) for i in range(1, 4000)]),
              ca.Graph.from_edges(2000, [(i, i + 1) for i in range(1999)]),
              exact_graph(rng, 180, 8000), none]
    for stream in (ca.STREAM_HASHED, ca.STREAM_REFERENCE):
        check(graphs, 5, stream, block=512, groups_per_cu=1, use_graph=True)


def test_repeated_edges_and_loops():
    # every neighbour relation stands in both rows, with different multiplicities, beside loops
    lists = [[1, 1, 1, 0], [0, 2], [1, 2, 3], [2, 2, 4], [3], [6], [5, 5]]
    check([rows(7, lists)], 3, ca.STREAM_HASHED)


def test_large_deviates_take_the_general_kernel():
    # beta 1e-5: deviates above 2^19 - 2 do not fit the packed keys
    rng = np.random.default_rng(4)
    check([exact_graph(rng, 300, 500)], 3, ca.STREAM_HASHED, beta=1e-5)
    check([exact_graph(rng, 300, 500)], 3, ca.STREAM_HASHED, beta=1e-4)
