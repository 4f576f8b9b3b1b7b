"""The extent of the finite boxes of a column, and the distances of dwithin
given as one number or as one per row."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from vibespatial_amd import join as J
from vibespatial_amd.api import GeoSeries
from vibespatial_amd.geometry import Point, PointArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 63, 64, 257, 512 * 256 + 1])
def test_extent_counts_finite_boxes_only(n):
    rng = np.random.default_rng(n)
    b = rng.normal(0, 1e6, (n, 4))
    b[:, 2:] = b[:, :2] + rng.uniform(0, 5, (n, 2))
    bad = rng.random(n) < 0.3
    b[bad, rng.integers(0, 4, n)[bad]] = rng.choice([np.nan, np.inf, -np.inf], n)[bad]
    ok = np.isfinite(b).all(axis=1)
    got = J.boxes_extent(torch.from_numpy(b).cuda())
    want = (np.inf, np.inf, -np.inf, -np.inf) if not ok.any() else (*b[ok, :2].min(0), *b[ok, 2:].max(0))
    assert got == (*want, int(ok.sum()))


def test_one_distance_equals_the_same_distance_per_row():
    rng = np.random.default_rng(3)
    q = [Point(*p) for p in rng.uniform(0, 10, (40, 2))] + [None, None]  # the points are the first rows
    tree = GeoSeries(PointArray(rng.uniform(0, 10, 200), rng.uniform(0, 10, 200))).sindex
    one = tree.query(GeoSeries(q), predicate="dwithin", distance=1.5)
    for dist in (np.float64(1.5), np.array([1.5]), np.full(42, 1.5)):
        assert np.array_equal(tree.query(GeoSeries(q), predicate="dwithin", distance=dist), one)
    assert one.shape[0] == 2 and one.dtype == np.int64 and one.shape[1] > 100
