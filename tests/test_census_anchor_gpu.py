"""The anchor pass of the pair census (census5_kernels.hip) at its edges --
windows of targets beginning and ending at a row's entries, targets below
the window, light anchors at their limits, out-degrees around a mask's
words -- against the per-edge kernels and closed forms."""
import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu


def _graph(n, edges):
    e = np.unique(np.sort(np.asarray(edges, dtype=np.int64), axis=1), axis=0)
    e = e[e[:, 0] != e[:, 1]]
    both = np.concatenate([e, e[:, ::-1]])
    both = both[np.lexsort((both[:, 1], both[:, 0]))]
    rp = np.zeros(n + 1, dtype=np.int64)
    rp[1:] = np.cumsum(np.bincount(both[:, 0], minlength=n))
    return ma.Graph.from_csr(rp, both[:, 1].astype(np.int32))


def _blocks(n, draws, blocks, seed):
    """Uniform edges, plus dense blocks of vertices scattered over the ids."""
    rng = np.random.default_rng(seed)
    edges = [rng.integers(0, n, (draws, 2))]
    for size in blocks:
        ids = rng.choice(n, size, replace=False)
        i, j = np.triu_indices(size, 1)
        keep = rng.random(len(i)) < 0.9
        edges.append(np.stack([ids[i[keep]], ids[j[keep]]], axis=1))
    return _graph(n, np.concatenate(edges))


@pytest.mark.parametrize("n,draws,blocks", [
    (1664, 9000, (20, 64)), (1665, 9000, (66, 130)), (3329, 30000, (70,)),
    (11649, 90000, (72, 145, 290)), (65537, 400000, (40, 66, 150)),
    (90001, 500000, (70, 140, 300))])
def test_windows_vs_kernels(gpu_available, n, draws, blocks):
    dg = ma.DeviceGraph(_blocks(n, draws, blocks, n), 0)
    for p in (2, 6):
        assert (dg.pattern_count(p)[0] == dg.pattern_count(
            p, ma.make_tune(pattern_census=-1))[0]), p
    dg.close()


@pytest.mark.parametrize("q", [3, 9, 11, 17, 63, 64, 65, 66, 129, 130, 257,
                               258, 513, 514])
@pytest.mark.parametrize("copies", [1, 140])
def test_cliques(gpu_available, q, copies):
    """Disjoint cliques hold no induced fork, star, bull or paw: every term
    cancels.  140 copies of q >= 513 lie across the window's lower end."""
    i, j = np.triu_indices(q, 1)
    if copies * len(i) > 10_000_000:
        copies = 128
    base = np.repeat(np.arange(copies) * q, len(i))
    edges = np.stack([base + np.tile(i, copies), base + np.tile(j, copies)],
                     axis=1)
    dg = ma.DeviceGraph(_graph(copies * q, edges), 0)
    got = {p: dg.pattern_count(p)[0] for p in (2, 3, 5, 6)}
    dg.close()
    assert got == {2: 0, 3: 0, 5: 0, 6: 0}
