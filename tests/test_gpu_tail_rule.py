"""Which graphs above 2^18 edge slots the one-workgroup tail takes: not the local variant's of more than 128 slots a
vertex, and above 4096 vertices none whose cut-off takes several hash parts to count against (11 808 edges do not).  A
call that runs in the tail launches no relabel.  Results against the oracle on both sides."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu

CASES = [  # vertices, edges, variant, cut-off, in the tail
    (1000, 131072, "local", 64, True), (1000, 140000, "local", 64, False), (2500, 160000, "local", 64, True),
    (2499, 160000, "local", 64, False), (4096, 180000, "exp", 60000, True), (4097, 180000, "exp", 60000, False),
    (4097, 180000, "exp", 11808, True), (4097, 180000, "exp", 11809, False), (8000, 131072, "exp", 60000, True),
    (8000, 220000, "exp", 64, True), (8000, 220000, "local", 60000, False)]


@pytest.mark.parametrize("n,m,variant,seq,tail", CASES)
def test_route(n, m, variant, seq, tail):
    rng = np.random.default_rng(n + m)
    keys = np.unique(rng.integers(0, n * n, size=4 * m))
    u, v = keys // n, keys % n
    ring = np.arange(n)
    keys = np.unique(np.minimum(u, v)[u != v] * n + np.maximum(u, v)[u != v])
    have = np.unique(np.minimum(ring, (ring + 1) % n) * n + np.maximum(ring, (ring + 1) % n))  # no isolated vertex
    keys = np.concatenate([have, rng.permutation(np.setdiff1d(keys, have))[: m - n]])
    assert len(keys) == m
    g = ca.Graph.from_edges(n, np.stack([keys // n, keys % n], 1))
    kw = dict(variant=variant, seed=5, seq_limit=seq)
    if variant == "exp":
        kw["stream"] = ca.STREAM_HASHED
    run = oracle.Run(g.offsets, g.targets, **kw)
    lv = run.levels()
    lab, st = ca.find_components(g, **kw)
    assert np.array_equal(lab, run.labels())
    assert (st["levels"], st["radius_sum"]) == (len(lv), sum(x[3] for x in lv))
    assert (st["kernel_launches"]["relabel"] == 0) == tail
