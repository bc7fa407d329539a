"""The relabel's two launches without labels in LDS, on both sides of 1024 blocks, against the oracle."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1023 * 256, 1024 * 256, 1024 * 256 + 1])
def test_relabel_launch_sizes(n):
    """A ring of short rows: the virtual blocks are the vertices' number by 256."""
    v = np.arange(n)
    g = ca.Graph.from_edges(n, np.stack([v, (v + 1) % n], 1))
    run = oracle.Run(g.offsets, g.targets, variant="exp", seed=3, seq_limit=0, stream=ca.STREAM_HASHED)
    dg = ca.DeviceGraph(g)
    lab, st = dg.find_components(variant="exp", seed=3, seq_limit=0, stream=ca.STREAM_HASHED, use_bfs=True)
    dg.close()
    lv = run.levels()
    assert np.array_equal(lab, run.labels())
    assert (st["levels"], st["radius_sum"]) == (len(lv), sum(x[3] for x in lv))
