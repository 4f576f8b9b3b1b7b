"""Polygons of several parts in the learned join, at the limits of its paths:
the staged-edge limit (512 edges) and the part-mask limit (32 parts)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from vibespatial_amd import join as J
from vibespatial_amd import synthetic as S
from vibespatial_amd.device import DevicePoints, DevicePolygons
from vibespatial_amd.geometry import PolygonArray

pytestmark = pytest.mark.gpu


def _parted(rng, n_rows, parts, vertices):
    """Rows of `parts` star parts each; neighbouring parts overlap, so a point
    may lie on the boundary of one part and inside another."""
    k = n_rows * parts
    row, part = np.repeat(np.arange(n_rows), parts), np.tile(np.arange(parts), n_rows)
    cx, cy = rng.uniform(0, 100, n_rows)[row] + 3.0 * part, rng.uniform(0, 100, n_rows)[row] + rng.uniform(-2, 2, k)
    p = S.star_polygons(rng, cx, cy, rng.uniform(2, 4, k), np.full(k, vertices))
    return PolygonArray(p.x, p.y, p.ring_offsets, p.part_offsets, np.arange(n_rows + 1) * parts)


@pytest.mark.parametrize("parts,vertices", [(2, 8), (2, 256), (2, 300), (31, 5), (32, 15), (32, 16), (32, 40), (33, 6),
                                            (40, 30)])
def test_rows_of_many_parts_match_oracle(parts, vertices):
    rng = np.random.default_rng(parts * 1000 + vertices)
    P = _parted(rng, 40, parts, vertices)
    v = rng.integers(0, len(P.x), 600)
    px = np.concatenate([rng.uniform(-5, 105 + 3 * parts, 6000), P.x[v]])
    py = np.concatenate([rng.uniform(-5, 105, 6000), P.y[v]])
    o = rng.permutation(len(px))
    px, py = px[o], py[o]
    Q = DevicePoints(torch.from_numpy(px).cuda(), torch.from_numpy(py).cuda())
    D = DevicePolygons.from_host(P)
    b = J.polygon_bounds(D)
    for pred in ("within", "intersects", "touches"):
        l, r, _ = J.sjoin_points_polygons_learned(Q, D, b, pred)
        el, er = oracle.sjoin_points_polygons(px, py, P, pred)
        assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er), pred
    idx = J.LearnedPointIndex(Q)
    for pred, same in (("contains", "within"), ("covers", "intersects"), ("touches", "touches")):
        l, r, _ = idx.query_polygons(D, b, pred)
        el, er = oracle.sjoin_points_polygons(px, py, P, same)
        k = np.lexsort((el, er))
        assert np.array_equal(l.cpu().numpy(), er[k]) and np.array_equal(r.cpu().numpy(), el[k]), pred
