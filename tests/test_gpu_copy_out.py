"""Labels copied out to pageable memory: every word written and none beside it, at the sizes where the copy
changes its way (helper threads above 256 KB, pieces of 64 k labels, or 128 k above the ring's 4 M, which
later transfers of 1 M go round; two, three or four bytes a label), into buffers at odd offsets, and from several threads at once (one
of them gets the pinned ring, the others copy the plain way)."""
import ctypes
import threading

import numpy as np
import pytest

import components_amd as ca

pytestmark = pytest.mark.gpu

SENTINEL = 0xABCD1234
U32P = ctypes.POINTER(ctypes.c_uint32)


def expected(n):
    ref = np.arange(n, dtype=np.uint32)
    ref[n - 1] = 0
    return ref


def graph(n):
    """One edge between the first and the last vertex: labels are the ids but for the last."""
    off = np.ones(n + 1, np.uint64)
    off[0] = 0
    off[n] = 2
    return ca.DeviceGraph(ca.Graph(off, np.array([n - 1, 0], np.uint32)))


def copy_into(fn, n, lead):
    buf = np.full(n + lead + 8, SENTINEL, np.uint32)
    fn(buf[lead:].ctypes.data_as(U32P))
    assert (buf[:lead] == SENTINEL).all() and (buf[lead + n:] == SENTINEL).all()
    assert np.array_equal(buf[lead:lead + n], expected(n))


KB = 1 << 8  # words per KB


@pytest.mark.parametrize("n", [2, 1000, 65536, 65537, 256 * KB - 1, 256 * KB, 256 * KB + 1, 1024 * KB, 1024 * KB + 1, 2048 * KB - 1, 2048 * KB, 2048 * KB + 1, 9000 * KB + 3,
                               16384 * KB - 1, 16384 * KB + 1, 20480 * KB, 20480 * KB + 1, 50000 * KB + 7, 1 << 24,
                               (1 << 24) + 1])
def test_every_word_and_no_other(n):
    g = graph(n)
    L = ca.lib()
    for lead in (0, 1, 3):
        def call(p):
            o = ca.options(seq_limit=0)
            assert L.kc_find_components(g.h, ctypes.byref(o), p, None) == ca.KC_OK
        copy_into(call, n, lead)
        copy_into(lambda p: L.kc_copy_labels(g.h, p), n, lead)
    g.close()


def test_several_threads():
    sizes = [3000 * KB, 700 * KB, 5000 * KB + 5, 40]
    graphs = [graph(n) for n in sizes]
    errors = []

    def work(g, n):
        try:
            for _ in range(6):
                lab, st = g.find_components(seq_limit=0)
                assert np.array_equal(lab, expected(n)) and st["components"] == n - 1
        except BaseException as e:  # noqa: BLE001 (reported below)
            errors.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(graphs, sizes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in graphs:
        g.close()
    assert not errors, errors


def test_refused_call_leaves_the_buffer():
    n = 1500 * KB
    g = graph(n)
    buf = np.full(n, SENTINEL, np.uint32)
    o = ca.options(variant="shortcut", replicate=True)
    assert ca.lib().kc_find_components(g.h, ctypes.byref(o), buf.ctypes.data_as(U32P), None) == ca.KC_ERR_UNSUPPORTED
    o = ca.options(seq_limit=0, max_levels=1, stream=ca.STREAM_HASHED)
    g2 = ca.DeviceGraph.generate("gnm_undirected", n=n, m=2 * n, seed=3)
    assert ca.lib().kc_find_components(g2.h, ctypes.byref(o), buf.ctypes.data_as(U32P), None) == ca.KC_ERR_INVALID
    assert (buf == SENTINEL).all()
    g.close()
    g2.close()
