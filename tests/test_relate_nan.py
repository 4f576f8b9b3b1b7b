"""The device relation of two polygonal rows compiled for the host: its answers
against the rational oracle, and its end on rows with non-finite coordinates
(the walk along an edge stopped at the edge's end point, which a NaN never
equals)."""

from __future__ import annotations

import itertools
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import relate_ref as R
from vibespatial_amd import _lib
from vibespatial_amd.geometry import MultiPolygon, Polygon, PolygonArray, box

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _args(P):
    return [a.ctypes.data for a in (P.x, P.y, P.geom_offsets, P.part_offsets, P.ring_offsets)]


def host_relation(A, a, B, b):
    """(interiors meet, a in b, b in a, boundaries meet)"""
    m = _lib.lib().vs_host_polygon_relation(*_args(A), a, *_args(B), b)
    return tuple(bool(m & k) for k in (1, 2, 4, 8))


def test_host_relation_matches_oracle():
    rng = np.random.default_rng(3)
    rows = []
    for _ in range(7):
        x, y, w, h = (*rng.integers(0, 6, 2), *rng.integers(2, 6, 2))
        rows += [box(x, y, x + w, y + h),
                 Polygon([(x, y), (x + w, y), (x + w, y + 1), (x + 1, y + 1), (x + 1, y + h), (x, y + h)])]
    rows += [Polygon([(0, 0), (9, 0), (9, 9), (0, 9)], [[(2, 2), (2, 6), (6, 6), (6, 2)]]),
             MultiPolygon([box(0, 0, 2, 2), box(4, 4, 7, 7)])]
    P = PolygonArray.from_geometries(rows)
    for i, j in itertools.product(range(len(rows)), repeat=2):
        meet, in_b, in_a, touch = host_relation(P, i, P, j)
        got = {"intersects": meet or touch, "within": in_b, "contains": in_a, "covers": in_a, "covered_by": in_b,
               "contains_properly": in_a and not touch, "touches": touch and not meet,
               "overlaps": meet and not in_a and not in_b}
        assert got == {p: R.predicate(p, P, i, P, j) for p in got}, (i, j)


def bad_rows(bad):
    """Three finite rows, then a square with one coordinate, or one point, bad."""
    rows = [box(0, 0, 8, 8), box(4, 4, 12, 12), box(8, 0, 12, 8)]
    for k, axes in itertools.product(range(4), ((0,), (1,), (0, 1))):
        ring = [[2.0, 2.0], [6.0, 2.0], [6.0, 6.0], [2.0, 6.0]]
        for a in axes:
            ring[k][a] = bad
        rows.append(Polygon([tuple(v) for v in ring]))
    return PolygonArray.from_geometries(rows)


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_non_finite_coordinates_end(bad):
    # in a process of its own, so that a walk without end fails instead of holding up the run
    code = f"""
import sys; sys.path.insert(0, {ROOT!r})
import itertools
from tests.test_relate_nan import bad_rows, host_relation
P = bad_rows(float({str(bad)!r}))
for i, j in itertools.product(range(len(P)), repeat=2):
    host_relation(P, i, P, j)
print("ended")
"""
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=90)
    assert done.returncode == 0 and "ended" in done.stdout, done.stderr


@pytest.mark.gpu
def test_device_relations_end_on_nan_rows():
    import torch

    from vibespatial_amd import api

    P = bad_rows(float("nan"))
    pairs = torch.tensor(list(itertools.product(range(len(P)), repeat=2)), dtype=torch.int64, device="cuda")
    l, r = pairs[:, 0].contiguous(), pairs[:, 1].contiguous()
    for pred in ("touches", "overlaps", "within", "covers", "contains_properly", "intersects"):
        for hl in (0, 1, 63):  # by product of the rows' sizes, one wave per pair, one thread per pair
            print(f"nan rows {pred} {hl}", flush=True)
            kl, kr = api._refine(1, pred, l, r, None, P, P, heavy_log2=hl)
            got = {(a, b) for a, b in zip(kl.tolist(), kr.tolist()) if a < 3 and b < 3}
            assert got == {(a, b) for a, b in itertools.product(range(3), repeat=2) if R.predicate(pred, P, a, P, b)}
