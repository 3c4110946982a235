"""The row passes of the census (census_rows.hip) at the edges of their
classes (64 / 256 / 704 out-neighbours), with more lower neighbours than one
chunk of columns holds, and with vertices below the bitmap's window, against
closed forms."""
from math import comb

import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu


def _from_rows(rows):
    rp = np.zeros(len(rows) + 1, dtype=np.int64)
    rp[1:] = np.cumsum([len(r) for r in rows])
    return ma.Graph.from_csr(rp, np.concatenate(rows).astype(np.int32))


@pytest.mark.parametrize("s", [64, 65, 66, 256, 257, 258, 704, 705, 706, 769])
def test_clique_with_pendants(gpu_available, s):
    """K_s with a pendant per vertex: out-degrees s - 1, s - 2, ..., 0."""
    rows = [np.concatenate([np.delete(np.arange(s), v), [s + v]])
            for v in range(s)] + [np.array([v]) for v in range(s)]
    dg = ma.DeviceGraph(_from_rows(rows), 0)
    want = {1: 0, 4: comb(s, 2), 7: 0, 8: 3 * s * comb(s - 1, 3)}
    got = {p: dg.pattern_count(p)[0] for p in want}
    dg.close()
    assert got == want


@pytest.mark.parametrize("s,m", [(2, 3000), (65, 63), (70, 64), (70, 2497),
                                 (257, 1300)])
def test_complete_split(gpu_available, s, m):
    """K_s joined to m independent vertices: the clique's vertices have all
    m below them, in one to four chunks of columns."""
    rows = [np.delete(np.arange(s + m), v) for v in range(s)]
    rows += [np.arange(s)] * m
    dg = ma.DeviceGraph(_from_rows(rows), 0)
    want = {1: s * comb(m, 3), 4: 0, 7: 2 * comb(s, 2) * comb(m, 3), 8: 0}
    got = {p: dg.pattern_count(p)[0] for p in want}
    dg.close()
    assert got == want


def test_below_the_window(gpu_available):
    """A random graph ranked below a triangle-free one of 66000 vertices
    counts what it counts alone (every bull, paw and clique is its own)."""
    n, half, d = 300, 33000, 130
    rng = np.random.default_rng(7)
    upper = np.triu(rng.random((n, n)) < 0.3, 1)
    rows = [np.flatnonzero(r) for r in upper | upper.T]
    assert max(map(len, rows)) < d
    alone = ma.DeviceGraph(_from_rows(rows), 0)
    left, j = np.arange(half)[:, None], np.arange(d)[None, :]
    rows += list(np.sort(n + half + (left + 7 * j) % half, axis=1))
    rows += list(np.sort(n + (left - 7 * j) % half, axis=1))
    both = ma.DeviceGraph(_from_rows(rows), 0)
    for p in (5, 6, 7, 8):
        want = alone.pattern_count(p)[0]
        assert want > 0 and both.pattern_count(p)[0] == want, p
    assert (both.pattern_count(1)[0] ==
            alone.pattern_count(1)[0] + 2 * half * comb(d, 3))
    assert both.tc_count()[0] == alone.tc_count()[0]


@pytest.mark.parametrize("m", [255, 256, 257, 1023, 1024, 1025])
def test_classes_by_lower_neighbours(gpu_available, m):
    """K_5 joined to m independent vertices: four out-neighbours or fewer at
    the edges of the classes by lower neighbours (256, 1024)."""
    s = 5
    rows = [np.delete(np.arange(s + m), v) for v in range(s)]
    rows += [np.arange(s)] * m
    dg = ma.DeviceGraph(_from_rows(rows), 0)
    want = {1: s * comb(m, 3), 4: 0, 7: 2 * comb(s, 2) * comb(m, 3), 8: 0}
    got = {p: dg.pattern_count(p)[0] for p in want}
    dg.close()
    assert got == want


@pytest.mark.parametrize("copies", [40, 4200])
@pytest.mark.parametrize("s,m", [(2, 1), (16, 8), (31, 2), (32, 1), (33, 1),
                                 (34, 1), (20, 13), (8, 31), (8, 33)])
def test_a_wave_per_vertex(gpu_available, s, m, copies):
    """Copies of K_s joined to m vertices: at most 32 neighbours above and
    below take a wave each where there are more than 4096 of them."""
    n = s + m
    rows = [np.delete(np.arange(n), v) for v in range(s)] + [np.arange(s)] * m
    block = np.concatenate(rows)
    rp = np.concatenate([[0], np.cumsum(np.tile([len(r) for r in rows],
                                                copies))])
    col = (block[None, :] + n * np.arange(copies)[:, None]).ravel()
    dg = ma.DeviceGraph(ma.Graph.from_csr(rp, col.astype(np.int32)), 0)
    want = {1: copies * s * comb(m, 3), 4: 0,
            7: 2 * copies * comb(s, 2) * comb(m, 3), 8: 0}
    got = {p: dg.pattern_count(p)[0] for p in want}
    dg.close()
    assert got == want
