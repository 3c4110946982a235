"""What mgpm_stats says of a triangle count against hub bitmaps: the ids that
it tests and the bytes that it has to read, from the DAG."""
import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu

HUBS, CHUNK = 65535, 8


def _expected(g):
    rp, ci = g.csr()
    n, deg = g.n, np.diff(rp)
    rank = np.empty(n, dtype=np.int64)
    rank[np.argsort(deg, kind="stable")] = np.arange(n)
    tail, head = np.repeat(rank, deg), rank[ci]
    up = head > tail
    arcs = np.sort(tail[up] * n + head[up])
    a, b = arcs // n, arcs % n
    out = np.bincount(a, minlength=n)
    hubs = np.bincount(a[b >= n - HUBS], minlength=n)
    past = np.cumsum(out)[a] - 1 - np.arange(len(a))
    chunks = -(-np.minimum(past, hubs[a]) // CHUNK)
    owner = (np.bincount(b, minlength=n) > 0) & (hubs > 0)
    rows = -(-hubs[owner] // CHUNK)
    return (CHUNK * int(chunks.sum()),
            16 * int(owner.sum()) + 8 * len(a)
            + 2 * CHUNK * int(chunks.sum() + rows.sum()))


@pytest.mark.parametrize("make", [
    lambda: ma.Graph.rmat(11, 32, seed=6),
    lambda: ma.Graph.rmat(18, 16, seed=7),
    lambda: ma.Graph.er(140003, 3000001, seed=8),
])
def test_stats_of_the_hub_path(gpu_available, make):
    g = make()
    dg = ma.DeviceGraph(g, 0)
    for _ in range(2):
        c, st = dg.tc_count()
        assert st.path == 3
        assert (st.probes, st.bytes_alg) == _expected(g)
    _, st = dg.tc_count(ma.make_tune(tc_layout=-1))
    assert st.path == 1
    assert st.bytes_alg == 8 * (st.n + 1) + 20 * st.m_plus + 4 * st.s_plus
    dg.close()
