"""Index queries sized by their plan: one scan where the bound is allocated,
two where it is not or where there is no memory for it, the empty query, few
rows, whose plan is not waited for, output that is sized by the pairs and not by
the scan, and the C entry that scans and finishes at one capacity."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from vibespatial_amd import _lib
from vibespatial_amd import join as J
from vibespatial_amd import synthetic as S
from vibespatial_amd.device import DevicePoints, DevicePolygons, ptr, stream
from vibespatial_amd.geometry import Polygon, PolygonArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limit", [2**28, 3000, 0])
@pytest.mark.parametrize("key_bytes", [4, 8])
def test_planned_queries_match_oracle(monkeypatch, limit, key_bytes):
    monkeypatch.setattr(J, "POSITION_LIMIT", limit)
    w = S.c1(n_points=30_000, n_polys=120)
    x, y, P = w.points.x, w.points.y, w.polygons
    idx = J.LearnedPointIndex(DevicePoints.from_host(w.points), key_bytes=key_bytes)
    D = DevicePolygons.from_host(P)
    b = J.polygon_bounds(D)
    el, er = oracle.sjoin_points_polygons(x, y, P, "within")
    o = np.lexsort((el, er))
    l, r, st = idx.query_polygons(D, b, "contains")
    assert np.array_equal(l.cpu().numpy(), er[o]) and np.array_equal(r.cpu().numpy(), el[o])
    assert st.scanned >= st.pairs and st.retries == (0 if limit > 3000 else 1)
    boxes = b.cpu().numpy()
    el, er = oracle.box_query_points(x, y, boxes)
    l, r, st = idx.query_boxes(b)
    assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er)
    # a row whose bounds are NaN has no pairs; no row at all has none either
    b[5] = float("nan")
    l, r, _ = idx.query_boxes(b)
    assert np.array_equal(l.cpu().numpy(), el[el != 5]) and np.array_equal(r.cpu().numpy(), er[el != 5])
    l, r, _ = idx.query_boxes(b[:0])
    assert l.numel() == 0 and r.numel() == 0


def test_few_hits_of_a_long_scan_leave_little_allocated():
    """Slivers across the map: their boxes hold most points, they hold few."""
    rng = np.random.default_rng(4)
    n, k = 400_000, 40
    x, y = rng.uniform(0, 100, n), rng.uniform(0, 100, n)
    a = rng.uniform(0, 20, (k, 2))
    P = PolygonArray.from_geometries([Polygon([tuple(v), (v[0] + 80.0, v[1] + 80.0), (v[0] + 80.1, v[1] + 80.0)])
                                      for v in a])
    idx = J.LearnedPointIndex(DevicePoints(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()))
    D = DevicePolygons.from_host(P)
    b = J.polygon_bounds(D)
    el, er = oracle.sjoin_points_polygons(x, y, P, "within")
    o = np.lexsort((el, er))
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    l, r, st = idx.query_polygons(D, b, "contains")
    peak = torch.cuda.max_memory_allocated() - before
    assert np.array_equal(l.cpu().numpy(), er[o]) and np.array_equal(r.cpu().numpy(), el[o])
    assert st.retries == 0 and st.scanned > 100 * st.pairs > 0
    assert l.untyped_storage().nbytes() == r.untyped_storage().nbytes() == 8 * len(el)
    assert peak < 10 * st.scanned  # the stage's 8 bytes a position, plan and output beside it
    l, r, st = idx.query_polygons(D, b, "touches")
    assert l.numel() == 0 and r.numel() == 0 and st.pairs == 0


def test_no_memory_for_the_bound_counts_first(monkeypatch):
    w = S.c1(n_points=300_000, n_polys=120)
    idx = J.LearnedPointIndex(DevicePoints.from_host(w.points))
    D = DevicePolygons.from_host(w.polygons)
    b = J.polygon_bounds(D)
    want = idx.query_polygons(D, b, "contains")

    def refuse_from(slots):  # no memory for a stage of that many slots
        limit = _lib.lib().vs_learned_scan_workspace_bytes(D.n_coords, slots)

        def ws(nbytes, dev):
            if nbytes >= limit:
                raise torch.OutOfMemoryError("no room")
            return torch.empty(max(int(nbytes), 1), dtype=torch.uint8, device=dev)

        monkeypatch.setattr(J, "_ws", ws)

    refuse_from(want[2].scanned)
    l, r, st = idx.query_polygons(D, b, "contains")
    assert st.retries == 1 and torch.equal(l, want[0]) and torch.equal(r, want[1])
    refuse_from(want[2].pairs)
    with pytest.raises(torch.OutOfMemoryError):
        idx.query_polygons(D, b, "contains")


@pytest.mark.parametrize("n_queries", [1, 15, 16, 17])
@pytest.mark.parametrize("few_slots", [2**20, 1200])
def test_few_queries(monkeypatch, n_queries, few_slots):
    """Either side of the rows from which the plan's scan length is read, with
    room for the pairs and without."""
    monkeypatch.setattr(J, "FEW_SLOTS", few_slots)
    w = S.c1(n_points=200_000, n_polys=120)
    x, y = w.points.x, w.points.y
    P = w.polygons.take(np.arange(n_queries))
    idx = J.LearnedPointIndex(DevicePoints.from_host(w.points))
    D = DevicePolygons.from_host(P)
    b = J.polygon_bounds(D)
    el, er = oracle.sjoin_points_polygons(x, y, P, "within")
    o = np.lexsort((el, er))
    l, r, st = idx.query_polygons(D, b, "contains")
    assert np.array_equal(l.cpu().numpy(), er[o]) and np.array_equal(r.cpu().numpy(), el[o])
    assert st.retries == int(n_queries <= J.FEW_QUERIES and len(el) > few_slots)
    el, er = oracle.box_query_points(x, y, b.cpu().numpy())
    l, r, st = idx.query_boxes(b)
    assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er)
    assert st.retries == int(n_queries <= J.FEW_QUERIES and len(el) > few_slots)


def test_pairs_are_complete_on_return():
    """As from every join: another stream may read them without waiting."""
    from vibespatial_amd import GeoSeries

    w = S.c1(n_points=2_000_000, n_polys=400)
    D = DevicePolygons.from_host(w.polygons)
    b = J.polygon_bounds(D)
    idx = J.LearnedPointIndex(DevicePoints.from_host(w.points))
    for _ in range(3):
        idx.query_polygons(D, b, "contains")
        assert torch.cuda.current_stream().query()
        idx.query_boxes(b)
        assert torch.cuda.current_stream().query()
    tree = GeoSeries(w.points).sindex
    rows = GeoSeries(w.polygons).values
    for k in range(3):
        tree.query(rows[k], predicate="contains", return_device=True)
        assert torch.cuda.current_stream().query()


@pytest.mark.parametrize("slots", [0, 1])
def test_scan_and_finish_at_one_capacity(slots):
    """vs_learned_query_run with room for the pairs, and with a slot too few."""
    w = S.c1(n_points=20_000, n_polys=90)
    idx = J.LearnedPointIndex(DevicePoints.from_host(w.points))
    b = J.polygon_bounds(DevicePolygons.from_host(w.polygons))
    el, er = oracle.box_query_points(w.points.x, w.points.y, b.cpu().numpy())
    cap = len(el) - slots
    L = _lib.lib()
    nq = int(b.shape[0])
    plan = torch.empty(L.vs_learned_plan_bytes(nq), dtype=torch.uint8, device="cuda")
    ws = torch.empty(L.vs_learned_run_workspace_bytes(0, cap), dtype=torch.uint8, device="cuda")
    pos, res = torch.zeros(1, dtype=torch.int64, device="cuda"), torch.zeros(16, dtype=torch.int64, device="cuda")
    l, r = (torch.full((cap,), -1, dtype=torch.int64, device="cuda") for _ in range(2))
    index = [ptr(idx.buf), idx.n, idx.key_bytes, idx.n_leaves, ptr(b)]
    _lib.check(L.vs_learned_query_plan(*index, None, None, None, nq, 0, ptr(pos), ptr(plan), plan.numel(), stream()),
               "plan")
    _lib.check(L.vs_learned_query_run(*index, None, None, None, None, None, nq, 0, 0, 0, _lib.PRED["intersects"], cap, 1,
                                      ptr(l), ptr(r), ptr(res), ptr(plan), plan.numel(), ptr(ws), ws.numel(),
                                      stream()), "run")
    assert int(res[1]) == len(el) <= int(pos)
    if slots == 0:
        assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er)
    else:
        assert bool((l == -1).all()) and bool((r == -1).all())
