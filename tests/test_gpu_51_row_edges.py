"""Point x polygon distances at the edge counts where the walk over a row
changes: groups of four and of 32 edges, rows from which one wave takes a pair
(257 coordinates), with a hole, a second part, and points on vertices, on edges,
inside, in the hole, and beyond, both ways round, against the oracle."""

from __future__ import annotations

import math

import numpy as np
import pytest

import oracle
from vibespatial_amd import GeoSeries
from vibespatial_amd.geometry import MultiPolygon, PointArray, Polygon, PolygonArray

pytestmark = pytest.mark.gpu


def _ring(n, r, cx, cy, rng):
    t = 2 * np.pi * np.arange(n) / n
    q = r * rng.uniform(0.85, 1.0, n)
    return list(zip((cx + q * np.cos(t)).tolist(), (cy + q * np.sin(t)).tolist()))


def _rows(n, rng):
    return PolygonArray.from_geometries([
        Polygon(_ring(n, 10.0, 0.0, 0.0, rng)),
        Polygon(_ring(max(n - 4, 3), 10.0, 30.0, 0.0, rng), [_ring(3, 4.0, 30.0, 0.0, rng)]),
        MultiPolygon([Polygon(_ring(max(n // 2, 3), 6.0, 0.0, 30.0, rng)),
                      Polygon(_ring(max(n - n // 2 - 2, 3), 6.0, 14.0, 30.0, rng), [_ring(4, 2.0, 14.0, 30.0, rng)])])])


def _points(P, rng, m):
    x, y = np.asarray(P.x), np.asarray(P.y)
    k = rng.integers(0, len(x) - 1, m)
    px = np.concatenate([x[k], (x[k] + x[k + 1]) / 2, rng.uniform(-15, 45, m), x[k] + 0.25, [0.0, 30.0, 14.0]])
    py = np.concatenate([y[k], (y[k] + y[k + 1]) / 2, rng.uniform(-15, 45, m), y[k], [0.0, 0.0, 30.0]])
    return PointArray(px, py)


@pytest.mark.parametrize("n", [3, 4, 5, 31, 32, 33, 34, 64, 65, 66, 254, 255, 256, 257, 258, 512, 700])
def test_row_edges(n):
    print(f"row edges n {n}", flush=True)
    rng = np.random.default_rng(n)
    P = _rows(n, rng)
    pts = _points(P, rng, 6 if n > 100 else 12)
    pb = np.stack([pts.x, pts.y, pts.x, pts.y], axis=1)
    gb = oracle.polygon_bounds(P)
    for d in (0.0, 0.25, 3.0, math.inf):
        for lk, rk, q, t, qb, tb in ((0, 1, pts, P, pb, gb), (1, 0, P, pts, gb, pb)):
            el, er = oracle.dwithin_pairs(lk, rk, q, t, np.full(len(qb), d), qb, tb)
            l, r = GeoSeries(t).sindex.query(GeoSeries(q).values, predicate="dwithin", distance=d)
            assert np.array_equal(l, el) and np.array_equal(r, er), (d, lk)
    for lk, rk, q, t in ((0, 1, pts, P), (1, 0, P, pts)):
        (l, r), dist = GeoSeries(t).sindex.nearest(GeoSeries(q).values, return_distance=True)
        el, er, ed = oracle.nearest_pairs(lk, rk, q, t)
        assert np.array_equal(l, el) and np.array_equal(r, er), lk
        assert np.array_equal(dist.view(np.int64), ed.view(np.int64)), lk
