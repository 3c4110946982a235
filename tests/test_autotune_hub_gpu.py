"""The autotuner where hub bitmaps win: what it returns counts as fast as a
call without a tune on the same handle, and its time is that path's."""
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu


def test_tuned_count_takes_the_winner(gpu_available):
    g = ma.Graph.rmat(16, 16, seed=5)  # tables 10 times as long
    dg = ma.DeviceGraph(g, 0)
    want, st = dg.tc_count()
    assert st.path == 3
    best, ms = dg.autotune(0, reps=2)
    c, st = dg.tc_count(best)
    assert c == want and st.path == 3
    c, st = dg.tc_count()
    assert c == want and st.path == 3
    # any other knob is a table plan's, and takes longer than the winner
    best.chunk_work //= 2
    c, st = dg.tc_count(best)
    assert c == want and st.path in (1, 2) and st.kernel_ms > ms
    # a handle that was not tuned takes the knobs at their word
    best.chunk_work *= 2
    other = ma.DeviceGraph(g, 0)
    c, st = other.tc_count(best)
    assert c == want and st.path in (1, 2)
    again, ms2 = dg.autotune(0, reps=2)  # a second tuning times tables too
    assert dg.tc_count(again)[1].path == 3 and ms2 > 0
    other.close()
    dg.close()
