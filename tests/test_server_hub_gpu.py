"""The server's budget and the hub plans of triangle counts: a plan is kept
where there is room for it and gives its memory back to a graph or a request
that needs it, so that what fits without the plans is served."""
import numpy as np
import pytest

import mercury_amd as ma

pytestmark = pytest.mark.gpu

SLACK = 1 << 17  # a lane's counters and rounding


def _graph(seed):
    return ma.Graph.rmat(15, 16, seed=seed)


@pytest.fixture(scope="module")
def sizes():
    """Bytes a graph keeps in a server without its hub plan, the plan's, a P2
    lane's workspace, and the graph's counts."""
    g = _graph(1)
    dg = ma.DeviceGraph(g, 0)
    p2 = dg.pattern_count(2)[0]
    before = dg.footprint()
    tc, st = dg.tc_count()
    hub = dg.footprint() - before
    assert st.path == 3 and hub > 8 * SLACK
    b = ma.Batch(0, lanes=1)
    b.run([(dg, 2)])
    work = b.footprint()
    b.close()
    dg.close()
    probe = ma.Server(0)
    probe.add_graph(g)
    base = probe.stats().resident_bytes - hub
    probe.close()
    return {"base": base, "hub": hub, "work": work, "tc": tc, "p2": p2}


def _server(budget):
    return ma.Server(0, slots=1, lanes=1, hbm_budget=budget)


def _count(srv, gid, pattern):
    r = srv.wait(srv.submit(gid, pattern))
    assert r.status == 0
    return r.count


def test_graph_without_room_for_its_hub_plan(gpu_available, sizes):
    srv = _server(sizes["base"] + SLACK)
    gid = srv.add_graph(_graph(1))
    resident = srv.stats().resident_bytes
    assert resident <= sizes["base"]
    for _ in range(3):
        assert _count(srv, gid, 0) == sizes["tc"]
    st = srv.stats()
    assert st.resident_bytes == resident
    assert st.resident_bytes + st.workspace_bytes <= st.budget_bytes
    srv.close()


def test_graph_takes_the_room_of_a_hub_plan(gpu_available, sizes):
    """The second graph needs half of what the first one's plan holds, while
    triangle counts of the first one are in flight."""
    srv = _server(2 * sizes["base"] + sizes["hub"] // 2 + SLACK)
    a = srv.add_graph(_graph(1))
    assert srv.stats().resident_bytes == sizes["base"] + sizes["hub"]
    tickets = [srv.submit(a, 0) for _ in range(200)]
    b = srv.add_graph(_graph(1))
    tickets += [srv.submit(b, 0) for _ in range(50)]
    for t in tickets:
        r = srv.wait(t)
        assert r.status == 0 and r.count == sizes["tc"]
    st = srv.stats()
    assert st.resident_bytes <= 2 * sizes["base"] + sizes["hub"] // 2
    assert st.resident_bytes + st.workspace_bytes <= st.budget_bytes
    with pytest.raises(ma.MgpmError) as ei:  # not without the plans either
        srv.add_graph(_graph(1))
    assert ei.value.code == -9
    assert _count(srv, a, 0) == _count(srv, b, 0) == sizes["tc"]
    srv.close()


def test_request_takes_the_room_of_a_hub_plan(gpu_available, sizes):
    srv = _server(sizes["base"] + sizes["work"] + sizes["hub"] // 2 + SLACK)
    gid = srv.add_graph(_graph(1))
    assert srv.stats().resident_bytes == sizes["base"] + sizes["hub"]
    assert _count(srv, gid, 0) == sizes["tc"]
    assert _count(srv, gid, 2) == sizes["p2"]
    assert srv.stats().resident_bytes == sizes["base"]
    assert _count(srv, gid, 0) == sizes["tc"]
    srv.close()


def test_graph_keeps_no_more_than_its_plans(gpu_available):
    """Beside the uploaded graph and its triangle plan, 12 bytes per CSR entry
    and 28 per vertex: the windows' offsets leave out vertices of one
    neighbour, and the uploaded CSR goes when its relabelled copy is there."""
    g = ma.Graph.rmat(17, 16, seed=4)
    dg = ma.DeviceGraph(g, 0)
    plans = dg.footprint()
    dg.pattern_count(2)
    before = dg.footprint()
    dg.tc_count()
    hub = dg.footprint() - before
    dg.close()
    srv = ma.Server(0)
    gid = srv.add_graph(g)
    kept = srv.stats().resident_bytes - hub
    assert kept <= plans + 12 * g.nnz + 28 * (g.n + 1)
    assert _count(srv, gid, 0) > 0
    srv.close()


def test_window_offsets_of_few_neighbours(gpu_available):
    """Heavy anchors whose neighbours have one neighbour, two or many."""
    rows, hubs, n = [], 6, 6 + 3000
    for h in range(hubs):  # a clique; leaf v hangs on hubs v % 6 (and v + 1)
        rows.append([x for x in range(hubs) if x != h])
    for v in range(hubs, n):
        mine = sorted({v % hubs, (v + 1) % hubs} if v % 3 == 0 else {v % hubs})
        rows.append(mine)
        for h in mine:
            rows[h].append(v)
    rp = np.zeros(n + 1, dtype=np.int64)
    rp[1:] = np.cumsum([len(r) for r in rows])
    g = ma.Graph.from_csr(rp, np.concatenate(rows).astype(np.int32))
    dg = ma.DeviceGraph(g, 0)
    for p in (2, 3, 5, 6):
        assert dg.pattern_count(p)[0] == dg.pattern_count(
            p, ma.make_tune(pattern_census=-1))[0], p
    dg.close()
