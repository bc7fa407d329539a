"""The batched form's persistent kernel, which takes the graphs of more than 8192 vertices: the size classes of the
smaller graphs run beside it."""
import pytest

import components_amd as ca

pytestmark = pytest.mark.gpu


def test_classes_run_beside_the_queue():
    def gnm(n, seed):
        return ca.generate("gnm_undirected", n=n, m=3 * n, seed=seed)

    large = [gnm(20001 + k, k + 1) for k in range(8)]
    small = [gnm(5000 + k, k + 1) for k in range(60)] * 60
    ms = []
    for graphs in (large, small, large + small):
        db = ca.DeviceBatch(ca.BatchGraphs.pack(graphs))
        db.set_tuning(block=256, groups_per_cu=4, use_graph=False)
        ms.append(sorted(db.run(seed=5, stream=ca.STREAM_HASHED, copy_labels=False)[1]["time_ms"] for _ in range(7))[3])
        db.close()
    print(f"queue {ms[0]:.2f} ms, classes {ms[1]:.2f} ms, both {ms[2]:.2f} ms", flush=True)
    assert ms[1] < ms[0]  # else the queue hides nothing
    assert ms[2] < ms[0] + 0.5 * ms[1]  # one after the other it is the sum
