"""Label copies around the size from which helper threads take part (262 144 labels): one thread moves whole words, or two
bytes a label where they fit, for one graph and for batches, whose labels are bounded by their largest graph."""
import numpy as np
import pytest

import components_amd as ca

pytestmark = pytest.mark.gpu

SIZES = [65535, 65536, 65537, 131073, 262143, 262144, 262145, 300001]


def pairs(n):
    """Neighbours 2k and 2k + 1 joined: every label is the even id."""
    off = np.minimum(np.arange(n + 1), n - n % 2).astype(np.uint64)
    tgt = np.arange(n - n % 2, dtype=np.uint32) ^ np.uint32(1)
    return ca.Graph(off, tgt), np.where(np.arange(n) < n - n % 2, np.arange(n) & ~1, np.arange(n)).astype(np.uint32)


@pytest.mark.parametrize("n", SIZES)
def test_one_graph(n):
    g, want = pairs(n)
    dg = ca.DeviceGraph(g)
    for variant in ("exp", "shortcut", "labels"):
        lab, st = dg.find_components(variant=variant)
        assert np.array_equal(lab, want) and st["components"] == len(np.unique(want))
        assert np.array_equal(dg.labels(), want)
    dg.close()


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("largest", [997, 65536, 65537])
def test_batch(n, largest):
    parts = [largest] * (n // largest) + ([n % largest] if n % largest > 1 else [])
    graphs = {k: pairs(k) for k in set(parts)}
    db = ca.DeviceBatch(ca.BatchGraphs.pack([graphs[k][0] for k in parts]))
    db.set_tuning(block=256, groups_per_cu=1, use_graph=False, split_vertices=8192)
    lab, _ = db.run(seed=3, stream=ca.STREAM_HASHED)
    db.close()
    assert np.array_equal(lab, np.concatenate([graphs[k][1] for k in parts]))
