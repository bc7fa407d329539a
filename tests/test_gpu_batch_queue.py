"""The batched form's persistent kernel, which takes the graphs of more than 8192 vertices (and, at a rate whose
deviates do not fit packed keys, all of them): launch shapes, replays of its captured launch with other seeds, a split
above the size classes.  Labels, levels and radii are compared with the oracle on each graph alone.  And the size
classes of the smaller graphs run beside it."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu

CLASS_VERTICES = 8192  # of the largest size class


def queued_batch():
    b = ca.batch_generate(graphs=36, log_n_min=11.0, log_n_max=14.6, seed=17)
    sizes = np.diff(b.vtx_off.astype(np.int64))
    assert (sizes > CLASS_VERTICES).sum() >= 12 and (sizes <= CLASS_VERTICES).sum() >= 12
    return b


def references(b, seed, **kw):
    out = []
    for k in range(b.graphs):
        g = b.graph(k)
        run = oracle.Run(g.offsets, g.targets, variant="exp", seed=seed, seq_limit=0, **kw)
        lv = run.levels()
        out.append((run.labels(), len(lv), sum(x[3] for x in lv)))
    return out


def compare(b, db, want, **kw):
    lab, _ = db.run(**kw)
    levels, _, radius = db.graph_stats()
    for k, (rl, rlev, rrad) in enumerate(want):
        assert np.array_equal(lab[int(b.vtx_off[k]):int(b.vtx_off[k + 1])], rl), (k, kw)
        assert (levels[k], radius[k]) == (rlev, rrad), (k, kw)


def test_launch_shapes():
    b = queued_batch()
    want = references(b, 3, stream=ca.STREAM_HASHED)
    db = ca.DeviceBatch(b)
    try:
        for block, groups, graph in [(256, 4, False), (256, 1, True), (512, 2, True), (1024, 1, False), (1024, 2, True),
                                     (256, 8, False)]:
            print(f"shape block={block} groups_per_cu={groups} graph={graph}", flush=True)
            db.set_tuning(block=block, groups_per_cu=groups, use_graph=graph)
            compare(b, db, want, seed=3, stream=ca.STREAM_HASHED)
    finally:
        db.close()


def test_reference_stream_and_level_cap():
    """The reference stream lets levels stall: the oracle takes up to 170 000 on these graphs.  Above the cap of 4096 a
    batch is refused, and the same handle then runs what stays below it."""
    b = queued_batch()
    want = references(b, 3, stream=ca.STREAM_REFERENCE)
    assert max(w[1] for w in want) > 4096
    db = ca.DeviceBatch(b)
    with pytest.raises(ca.KcError, match="level cap reached"):
        db.run(seed=3, stream=ca.STREAM_REFERENCE)
    compare(b, db, references(b, 3, stream=ca.STREAM_HASHED), seed=3, stream=ca.STREAM_HASHED)
    db.close()
    below = [k for k, w in enumerate(want) if w[1] <= 4096]
    part = ca.BatchGraphs.pack([b.graph(k) for k in below])
    assert (np.diff(part.vtx_off.astype(np.int64)) > CLASS_VERTICES).any()
    db = ca.DeviceBatch(part)
    compare(part, db, [want[k] for k in below], seed=3, stream=ca.STREAM_REFERENCE)
    db.close()


def test_replays_with_other_seeds():
    b = queued_batch()
    want = {seed: references(b, seed, stream=ca.STREAM_HASHED) for seed in (1, 2, 3)}
    db = ca.DeviceBatch(b)
    try:
        for rep in range(3):
            for seed in (3, 1, 2):
                db.set_tuning(block=256, groups_per_cu=4, use_graph=True)
                compare(b, db, want[seed], seed=seed, stream=ca.STREAM_HASHED)
                if rep == 1:  # eager work in between
                    db.set_tuning(block=256, groups_per_cu=4, use_graph=False)
                    compare(b, db, want[1], seed=1, stream=ca.STREAM_HASHED)
    finally:
        db.close()


def test_splits_above_the_classes():
    b = queued_batch()
    sizes = np.diff(b.vtx_off.astype(np.int64))
    want = references(b, 9, stream=ca.STREAM_HASHED)
    split = int(np.sort(sizes)[-4])  # three graphs on the device-wide path, the queue keeps the others
    assert split > CLASS_VERTICES
    db = ca.DeviceBatch(b)
    try:
        for graph in (False, True):
            for sp in (split, 0, CLASS_VERTICES):
                print(f"split={sp} graph={graph}", flush=True)
                db.set_tuning(block=512, groups_per_cu=1, use_graph=graph, split_vertices=sp)
                lab, _ = db.run(seed=9, stream=ca.STREAM_HASHED)
                levels, _, radius = db.graph_stats()
                for k, (rl, rlev, rrad) in enumerate(want):
                    assert np.array_equal(lab[int(b.vtx_off[k]):int(b.vtx_off[k + 1])], rl), (sp, k)
                    if not sp or sizes[k] <= sp:
                        assert (levels[k], radius[k]) == (rlev, rrad), (sp, k)
    finally:
        db.close()


def test_small_rate_queues_every_graph():
    # beta 6.9e-5: deviates reach 2^19 - 2 and more
    b = ca.batch_generate(graphs=40, log_n_min=2, log_n_max=11, seed=5)
    db = ca.DeviceBatch(b)
    try:
        for seed in (4, 5):
            want = references(b, seed, stream=ca.STREAM_HASHED, beta=6.9e-5)
            for graph in (True, False, True):
                db.set_tuning(block=256, groups_per_cu=2, use_graph=graph)
                compare(b, db, want, seed=seed, stream=ca.STREAM_HASHED, beta=6.9e-5)
    finally:
        db.close()


def test_autotune_leaves_a_shape_that_nothing_uses():
    b = ca.batch_generate(graphs=64, log_n_min=5, log_n_max=10, seed=3)
    want = references(b, 5, stream=ca.STREAM_HASHED)
    db = ca.DeviceBatch(b)
    try:
        db.set_tuning(block=512, groups_per_cu=3, use_graph=False)  # three groups are no candidate of the search
        t = db.autotune(seed=5, stream=ca.STREAM_HASHED)
        assert (t["block"], t["groups_per_cu"]) == (512, 3)
        compare(b, db, want, seed=5, stream=ca.STREAM_HASHED)
    finally:
        db.close()


def test_autotune_of_queued_graphs():
    b = queued_batch()
    want = references(b, 5, stream=ca.STREAM_HASHED)
    db = ca.DeviceBatch(b)
    try:
        t = db.autotune(seed=5, stream=ca.STREAM_HASHED)
        assert t["block"] in (256, 512, 1024) and t["groups_per_cu"] in (1, 2, 4, 8)
        lab, st = db.run(seed=5, stream=ca.STREAM_HASHED)
        assert st["tuning"]["split_vertices"] == t["split_vertices"]
        for k, w in enumerate(want):
            assert np.array_equal(lab[int(b.vtx_off[k]):int(b.vtx_off[k + 1])], w[0]), k
    finally:
        db.close()


def test_classes_run_beside_the_queue():
    def gnm(n, seed):
        return ca.generate("gnm_undirected", n=n, m=3 * n, seed=seed)

    large = [gnm(20001 + k, k + 1) for k in range(8)]
    small = [gnm(5000 + k, k + 1) for k in range(60)] * 60
    ms = []
    for graphs in (large, small, large + small):
        db = ca.DeviceBatch(ca.BatchGraphs.pack(graphs))
        db.set_tuning(block=256, groups_per_cu=4, use_graph=False)
        ms.append(min(db.run(seed=5, stream=ca.STREAM_HASHED, copy_labels=False)[1]["time_ms"] for _ in range(9)))
        db.close()
    print(f"queue {ms[0]:.2f} ms, classes {ms[1]:.2f} ms, both {ms[2]:.2f} ms", flush=True)
    assert ms[1] < ms[0]  # else the queue hides nothing
    assert ms[2] < ms[0] + 0.5 * ms[1]  # one after the other it is the sum
