"""Triangle counts against hub bitmaps (tc_hub.hip), the default path where
hubs dominate: the sizes around the 65535 hubs, rows longer than a wave's
chunks, owners with more partners than a batch of records, triangles without
a hub, batches, and calls in a row, against closed forms and the table
plans."""
from math import comb

import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu

HUB = 3  # Stats.path of the hub plan


def _graph(rows):
    rp = np.zeros(len(rows) + 1, dtype=np.int64)
    rp[1:] = np.cumsum([len(r) for r in rows])
    return ma.Graph.from_csr(rp, np.concatenate(rows).astype(np.int32))


def _same(g, want=None, hub=True):
    dg = ma.DeviceGraph(g, 0)
    c, st = dg.tc_count()
    assert (st.path == HUB) == hub
    table, ts = dg.tc_count(ma.make_tune(tc_layout=-1))
    assert c == table and ts.path == 1
    assert c == dg.tc_count()[0]
    if want is not None:
        assert c == want
    b = ma.Batch(0)
    assert b.run([(dg, 0), (dg, 0)])[0] == [c, c]
    b.close()
    dg.close()


@pytest.mark.parametrize("n,draws", [(260, 30000), (65534, 500000),
                                     (65535, 500000), (65536, 500000),
                                     (65537, 500000), (140003, 3000001)])
def test_er_around_the_hubs(gpu_available, n, draws):
    _same(ma.Graph.er(n, draws, seed=n))


@pytest.mark.parametrize("s", [181, 182, 512, 513, 520, 1030])
def test_complete(gpu_available, s):
    rows = [np.delete(np.arange(s), v) for v in range(s)]
    _same(_graph(rows), comb(s, 3), hub=s * (s - 1) // 2 >= 16384)


@pytest.mark.parametrize("s,m", [(2, 8192), (3, 5462), (9, 4097),
                                 (65, 400), (70, 70000)])
def test_complete_split(gpu_available, s, m):
    """K_s joined to m independent vertices, which are its partners."""
    rows = [np.delete(np.arange(s + m), v) for v in range(s)]
    rows += [np.arange(s)] * m
    _same(_graph(rows), comb(s, 3) + m * comb(s, 2))


@pytest.mark.parametrize("s", [2, 3, 17, 60])
def test_cliques_below_the_hubs(gpu_available, s):
    """Cliques ranked below 66000 triangle-free vertices: none of their
    triangles has a hub."""
    half, d, copies = 33000, 61, 5
    rows = [np.delete(np.arange(s), v) + s * c for c in range(copies)
            for v in range(s)]
    n = len(rows)
    left, j = np.arange(half)[:, None], np.arange(d)[None, :]
    rows += list(np.sort(n + half + (left + 7 * j) % half, axis=1))
    rows += list(np.sort(n + (left - 7 * j) % half, axis=1))
    _same(_graph(rows), copies * comb(s, 3))


def test_edges_only(gpu_available):
    """No arc follows another: no owner, nothing to count."""
    n = 40000
    _same(_graph([np.array([v ^ 1]) for v in range(n)]), 0)


def test_without_hubs_the_table_plan_counts(gpu_available):
    g = ma.Graph.er(1 << 20, 1 << 21, seed=3)
    dg = ma.DeviceGraph(g, 0)
    c, st = dg.tc_count()
    assert st.path != HUB
    assert c == dg.tc_count(ma.make_tune(tc_layout=-1))[0]
    dg.close()
