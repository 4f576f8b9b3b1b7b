"""Index queries sized by their plan: one scan where the bound is allocated,
two where it is not, and the empty query."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from vibespatial_amd import join as J
from vibespatial_amd import synthetic as S
from vibespatial_amd.device import DevicePoints, DevicePolygons

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
