"""Recorded batches whose triangle counts go against hub bitmaps: every replay
equals the single calls, with the program's own counts between replays."""
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu


def test_replays_with_hub_counts(gpu_available):
    dgs = [ma.DeviceGraph(ma.Graph.rmat(s, 16, seed=60 + s), 0)
           for s in (9, 12, 13, 16)]
    paths = [dg.tc_count()[1].path == 3 for dg in dgs]
    assert paths == [False, True, True, True]
    queries = [(dg, p) for dg in dgs for p in (0, 1, 0)]
    single = [dg.pattern_count(p)[0] for dg, p in queries]
    b = ma.Batch(0, lanes=4, use_graph=True)
    for r in range(5):
        counts, st = b.run(queries)
        assert counts == single and st.path == 101, r
        assert dgs[r % 4].tc_count()[0] == single[3 * (r % 4)]
    b.close()
    for dg in dgs:
        dg.close()
