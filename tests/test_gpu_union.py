"""Union-find components (the base case, the shortcuts variant, the allocation-free shortcuts) at the
sizes where the edge slots of one wave (512) and the search of a slot's row can go wrong: fewer, as
many and more slots than one wave's; rows far longer; long runs of empty rows inside one wave's
range; paths in index order and against it (the deepest trees); both sides of the second shortening
pass (2^16 vertices) and of the hook rounds (2^14 and 2^20 vertices, 16 slots a vertex).  Labels are exact: compared with the oracle's union-find."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu


def path(n):
    return ca.Graph.from_edges(n, np.stack([np.arange(n - 1), np.arange(1, n)], 1))


def shuffled(g, seed):
    rng = np.random.default_rng(seed)
    p = rng.permutation(g.n)
    src = np.repeat(np.arange(g.n), np.diff(g.offsets).astype(np.int64))
    return ca.Graph.from_edges(g.n, np.stack([p[src], p[g.targets]], 1))


def cases():
    rng = np.random.default_rng(11)
    out = {f"path{n}": path(n) for n in (2, 256, 257, 258, 16383, 70000, (1 << 20) + 1)}
    out["path_reversed_ids"] = shuffled(path(70000), 1)
    out["zigzag"] = ca.Graph.from_edges(4096, [(i, 4095 - i) for i in range(2048)] +
                                        [(4095 - i, i + 1) for i in range(2047)])
    out["star"] = ca.Graph.from_edges(5001, [(5000, i) for i in range(5000)])
    # 60000 empty rows between the two ends of single edges: one wave's slots span them all
    out["far_ends"] = ca.Graph.from_edges(60002, [(0, 60001), (1, 60000), (30000, 30001)])
    e = rng.integers(0, 200000, size=(300, 2))
    out["sparse_islands"] = ca.Graph.from_edges(200000, e)
    out["random"] = ca.Graph.from_edges(65536, rng.integers(0, 65536, size=(60000, 2)))
    out["dense"] = ca.Graph.from_edges(20000, rng.integers(0, 20000, size=(200000, 2)))
    out["hubs"] = ca.Graph.from_edges(30000, [(7, i) for i in range(8, 12000)] + [(20000, i) for i in range(20001, 30000)]
                                      + [(11999, 20500)])
    return out


@pytest.mark.parametrize("name,g", list(cases().items()))
def test_union_labels_match_oracle(name, g):
    ref = oracle.canonical_labels(g.offsets, g.targets)
    roots = int(np.sum(ref == np.arange(g.n)))
    dg = ca.DeviceGraph(g)
    print(f"union {name}: n={g.n} m={g.m}", flush=True)
    for kw in (dict(variant="shortcut"), dict(variant="exp", seq_limit=1 << 40),
               dict(variant="exp", seed=3, pre_contract="single", pre_blocks=3, seq_limit=0, stream=ca.STREAM_HASHED)):
        lab, st = dg.find_components(**kw)
        assert np.array_equal(lab, ref), (name, kw)
        assert st["components"] == roots, (name, kw)
    dg.close()
