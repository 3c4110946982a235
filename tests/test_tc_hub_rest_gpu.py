"""Triangles without a hub where the highest-ranked vertices have no arcs among
them (tc_hub.hip, hub_rest): lists of vertices ranked just below the hubs are
empty and begin where the DAG's columns end."""
from math import comb

import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu

HUBS, LOW, PART, K = 65535, 20, 100_000, 10


def _graph(extra):
    """10000 cliques of K; every one of the 65535 last vertices joined to ten
    cliques, in turn, and the LOW before them, below the hubs, all to the
    first ten cliques.  extra: pendant pairs, ranked first, for the number of
    arcs."""
    v = np.arange(PART)
    pairs = [np.stack([v[v % K < K - j], v[v % K < K - j] + j])
             for j in range(1, K)]
    first = PART + LOW
    hub = np.repeat(np.arange(HUBS), 100)
    pairs.append(np.stack([(np.arange(100 * HUBS)) % PART, first + hub]))
    pairs.append(np.stack([np.tile(np.arange(100), LOW),
                           PART + np.repeat(np.arange(LOW), 100)]))
    n = first + HUBS
    e = n + 2 * np.arange(extra)
    pairs.append(np.stack([e, e + 1]))
    n += 2 * extra
    a, b = np.concatenate(pairs, axis=1)
    key = np.sort(np.concatenate([a * n + b, b * n + a]))
    rp = np.zeros(n + 1, dtype=np.int64)
    rp[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    return ma.Graph.from_csr(rp, (key % n).astype(np.int32))


@pytest.mark.parametrize("align", [True, False])
def test_hubs_without_arcs_among_them(gpu_available, align):
    """align: the number of arcs is a multiple of 64, so that nothing pads the
    columns."""
    m = PART * (K - 1) // 2 + 100 * (HUBS + LOW)
    extra = -m % 64 + (0 if align else 1)
    g = _graph(extra)
    assert g.nnz == 2 * (m + extra)
    cliques = PART // K
    want = cliques * comb(K, 3) + (HUBS + LOW) * 10 * comb(K, 2)
    dg = ma.DeviceGraph(g, 0)
    c, st = dg.tc_count()
    assert st.path == 3 and c == want
    table, ts = dg.tc_count(ma.make_tune(tc_layout=-1))
    assert ts.path == 1 and table == want
    dg.close()
