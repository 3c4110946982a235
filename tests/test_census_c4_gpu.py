"""The 4-cycle pass of the census (census_c4.hip) where its kinds and classes
meet -- pairs above, across and below the counters' window, light and heavy
owners, a hub with more middles than 16 bits count -- against closed forms
and the per-edge kernels."""
from math import comb

import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu


def _bipartite(a, b, copies):
    """`copies` disjoint K_{a,b}."""
    block = [np.arange(a, a + b)] * a + [np.arange(a)] * b
    rows = [r + c * (a + b) for c in range(copies) for r in block]
    rp = np.zeros(len(rows) + 1, dtype=np.int64)
    rp[1:] = np.cumsum([len(r) for r in rows])
    return ma.Graph.from_csr(rp, np.concatenate(rows).astype(np.int32))


@pytest.mark.parametrize("a,b,copies", [
    (2, 2, 1), (3, 5, 1), (22, 24, 3),   # one owner class each
    (23, 24, 3), (30, 30, 1200),         # light and heavy across the window
    (2, 70000, 1)])                      # 32-bit counters, two rounds
def test_complete_bipartite(gpu_available, a, b, copies):
    """Complete bipartite graphs hold no induced path, fork, bull or paw."""
    dg = ma.DeviceGraph(_bipartite(a, b, copies), 0)
    stars = lambda k: copies * (a * comb(b, k) + b * comb(a, k))
    want = {1: stars(3), 2: 0, 3: 4 * stars(4) + 3 * stars(3), 4: 0, 5: 0,
            6: 0}
    got = {p: dg.pattern_count(p)[0] for p in want}
    dg.close()
    assert got == {p: w % 2**64 for p, w in want.items()}


@pytest.mark.parametrize("n,draws", [(65536, 300000), (65537, 300000),
                                     (70001, 420007), (300007, 900001)])
def test_window_edges(gpu_available, n, draws):
    dg = ma.DeviceGraph(ma.Graph.er(n, draws, seed=n), 0)
    for p in (2, 4):
        assert (dg.pattern_count(p)[0] == dg.pattern_count(
            p, ma.make_tune(pattern_census=-1))[0]), p
    dg.close()


@pytest.mark.parametrize("c,d", [(2, 40), (15, 40), (16, 40), (255, 260),
                                 (256, 260)])
def test_counter_widths(gpu_available, c, d):
    """Owners below the window with c middles (4, 8 and 16-bit counters take
    up to 15, 255 and more) on a bipartite graph whose left vertex x sees
    the right vertices x + 7j, j < d: owner i sees the left vertices i + 7j,
    j < c, so i and the right vertex i + 7m have as many common neighbours as
    m has sums j + k with j < c and k < d."""
    half, owners = 33000, 4
    x, j = np.arange(half)[:, None], 7 * np.arange(d)[None, :]
    left = [np.sort(r) for r in owners + half + (x + j) % half]
    right = [np.sort(r) for r in owners + (x - j) % half]
    for i in range(owners):
        for k in range(c):
            left[i + 7 * k] = np.concatenate([[i], left[i + 7 * k]])
    rows = [owners + i + 7 * np.arange(c) for i in range(owners)]
    rows += left + right
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    dg = ma.DeviceGraph(
        ma.Graph.from_csr(rp, np.concatenate(rows).astype(np.int32)), 0)
    got = dg.pattern_count(4)[0]
    dg.close()
    sums = np.bincount((np.arange(c)[:, None] + np.arange(d)).ravel())
    cycles = (half * sum(comb(d - k, 2) for k in range(1, d)) +
              owners * sum(comb(int(s), 2) for s in sums))
    paths = ((half * d - owners * c * d) * (d - 1) ** 2 +
             owners * c * d * d * (d - 1) + owners * c * (c - 1) * d)
    assert got == paths - 4 * cycles
