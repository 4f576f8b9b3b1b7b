"""The nearest bound's walk, 16 lanes to a query, at the tree sizes where its
steps end: one level of items, last groups of one and of 15, three and four
levels, a query count that leaves lanes over, against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from vibespatial_amd import GeoSeries
from vibespatial_amd import synthetic as S
from vibespatial_amd.geometry import PointArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 255, 256, 257, 4095, 4097])
@pytest.mark.parametrize("m", [1, 5, 67])
def test_bound_walk(n, m):
    print(f"bound walk items {n} queries {m}", flush=True)
    rng = np.random.default_rng(100 * n + m)
    q = PointArray(rng.uniform(-2e3, 3e3, m), rng.uniform(-2e3, 3e3, m))
    lattice = PointArray(rng.integers(0, 40, n) * 25.0, rng.integers(0, 40, n) * 25.0)  # ties, equal points
    near = PointArray(np.round(q.x / 12.5) * 12.5, np.round(q.y / 12.5) * 12.5)
    rows = S.star_polygons(rng, rng.uniform(0, 1000, n), rng.uniform(0, 1000, n), rng.uniform(2, 20, n),
                           rng.integers(3, 40, n))
    for t, kind in ((lattice, 0), (rows, 1)):
        for query in (q, near):
            (l, r), d = GeoSeries(t).sindex.nearest(GeoSeries(query).values, return_distance=True)
            el, er, ed = oracle.nearest_pairs(0, kind, query, t)
            assert np.array_equal(l, el) and np.array_equal(r, er), kind
            assert np.array_equal(d.view(np.int64), ed.view(np.int64)), kind
