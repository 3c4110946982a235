"""Batches of several threads on graphs that nothing has been counted on yet:
the census graph and the hub plan are built once, and every count is the
single call's."""
import threading

import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("patterns", [(0,), (0, 1, 7, 2)])
def test_batches_of_four_threads(gpu_available, patterns):
    graphs = [ma.Graph.rmat(12 + i % 2, 16, seed=50 + i) for i in range(6)]
    want = []
    for g in graphs:
        dg = ma.DeviceGraph(g, 0)
        want += [dg.pattern_count(p)[0] if p else dg.tc_count()[0]
                 for p in patterns]
        dg.close()
    dgs = [ma.DeviceGraph(g, 0) for g in graphs]
    queries = [(dg, p) for dg in dgs for p in patterns]
    got, start = [None] * 4, threading.Barrier(4)

    def work(k):
        b = ma.Batch(0, lanes=2)
        start.wait()
        got[k] = b.run(queries)[0]
        b.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == [want] * 4
    for dg in dgs:
        dg.close()
