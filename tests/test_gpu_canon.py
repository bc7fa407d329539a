"""Minimum ids per component: level sizes around a wave, a block and a step of four blocks' vertices, one component
beside many small ones in every mixture of lanes."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 65, 257, 2047, 2049, 8193, 300001])
@pytest.mark.parametrize("share", [0.0, 0.02, 0.5, 0.98, 1.0])
def test_mixed_components(n, share):
    """A giant component on a random share of the vertices, pairs elsewhere; the giant's first vertex last in rows."""
    rng = np.random.default_rng(n)
    perm = rng.permutation(n)
    k = int(round(share * n))
    giant, rest = perm[:k], perm[k:]
    e = [np.stack([giant[:-1], giant[1:]], 1)] if k > 1 else []
    p = rest[: len(rest) // 2 * 2].reshape(-1, 2)
    e.append(p)
    e = np.sort(np.concatenate(e), 1)
    g = ca.Graph.from_edges(n, e)
    want = oracle.Run(g.offsets, g.targets, variant="exp", seed=1, seq_limit=0, stream=ca.STREAM_HASHED).labels()
    for kw in (dict(variant="exp", use_bfs=True, stream=ca.STREAM_HASHED), dict(variant="local")):
        lab, st = ca.find_components(g, seed=1, seq_limit=0, record_trace=True, **kw)[:2]
        assert np.array_equal(lab, want)
        assert st["components"] == len(np.unique(want))
