"""Vertices of more than 704 out-neighbours, whose bit rows lie in the
workgroups' slabs (census_rows.hip): what the passes allocate, and the pass
over cliques with more lower neighbours than the rows hold columns for."""
from math import comb

import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu


def _join(s, m):
    """K_s joined to m independent vertices."""
    rows = [np.delete(np.arange(s + m), v) for v in range(s)]
    rows += [np.arange(s)] * m
    rp = np.zeros(len(rows) + 1, dtype=np.int64)
    rp[1:] = np.cumsum([len(r) for r in rows])
    return ma.Graph.from_csr(rp, np.concatenate(rows).astype(np.int32))


@pytest.mark.parametrize("pattern", [1, 4])
def test_no_triangle_lists_without_cliques(gpu_available, pattern):
    s = 900
    dg = ma.DeviceGraph(_join(s, 0), 0)
    b = ma.Batch(0, lanes=1)
    assert b.run([(dg, pattern)])[0] == [0]
    # A count per arc, and 256 workgroups of rows (15 words a neighbour) and
    # counts; the lists would be 12 bytes for each of C(900, 2) pairs.
    assert b.footprint() < 4 * comb(s, 2) + 256 * s * (15 * 8 + 8) + (1 << 20)
    b.close()
    dg.close()


@pytest.mark.parametrize("s,m", [(706, 513), (769, 600), (769, 1025)])
def test_more_lower_neighbours_than_columns(gpu_available, s, m):
    """The m independent vertices rank below the clique: m columns for each of
    its vertices, 512 at a time in the slab."""
    dg = ma.DeviceGraph(_join(s, m), 0)
    want = {1: s * comb(m, 3), 4: 0, 7: 2 * comb(s, 2) * comb(m, 3), 8: 0}
    got = {p: dg.pattern_count(p)[0] for p in want}
    dg.close()
    assert got == {p: c % 2**64 for p, c in want.items()}
