"""The one-wave-per-pair edge search at the sizes of its lists, tiles and queue:
rows of n edges that run close together without meeting, meeting in one point,
crossing in one place, nested, and inside a hole.  The relations are known by
construction; the one-thread route gets the same pairs."""

from __future__ import annotations

import numpy as np
import pytest

from vibespatial_amd.geometry import Polygon, PolygonArray

pytestmark = pytest.mark.gpu


def _zigzag(n, lift, close, low=None):
    """Ring whose n edges zigzag between y = lift and lift + 1; vertex `low`
    = (k, y) is moved to that y."""
    y = [lift + (k % 2) for k in range(n + 1)]
    if low is not None:
        y[low[0]] = low[1]
    return Polygon([(float(k), y[k]) for k in range(n + 1)] + [(float(n), close), (0.0, close)])


def _circle(n, r, cx=0.0, cy=0.0):
    t = 2 * np.pi * np.arange(n) / n
    return list(zip((cx + r * np.cos(t)).tolist(), (cy + r * np.sin(t)).tolist()))


@pytest.mark.parametrize("n", [15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 200, 700])
def test_close_rows(n):
    import torch

    from vibespatial_amd import api

    mid = (n // 2) & ~1
    A = PolygonArray.from_geometries([
        _zigzag(n, 0.0, -5.0), _zigzag(n, 0.0, -5.0), _zigzag(n, 0.0, -5.0), _zigzag(n, 0.0, -5.0),
        Polygon(_circle(n, 10.0)), Polygon(_circle(n, 10.0)), Polygon(_circle(n + 3, 99.0))])
    B = PolygonArray.from_geometries([
        _zigzag(n, 0.25, 9.0), _zigzag(n, 0.25, 9.0, (mid, 0.0)), _zigzag(n, 0.25, 9.0, (mid, -0.125)),
        _zigzag(2 * n + 1, 0.25, 9.0),
        Polygon(_circle(n + 1, 100.0)), Polygon(_circle(n + 1, 100.0), [_circle(n + 2, 50.0)]),
        Polygon(_circle(2 * n, 100.0), [_circle(n, 50.0)])])
    pairs = [(i, i) for i in range(7)]
    # per pair: apart, one common point, crossing, apart, inside, inside the hole,
    # and over the hole (inside the shell or crossing it, as n decides)
    expect = {"intersects": {1, 2, 4, 6}, "touches": {1}, "within": {4}, "covered_by": {4}, "contains": set(),
              "contains_properly": set()}
    l = torch.tensor([p[0] for p in pairs], dtype=torch.int64, device="cuda")
    r = torch.tensor([p[1] for p in pairs], dtype=torch.int64, device="cuda")
    for pred, want in expect.items():
        for hl in (0, 1, 63):
            kl, _ = api._refine(1, pred, l, r, None, A, B, heavy_log2=hl)
            assert set(kl.cpu().tolist()) - {6} == want - {6}, (pred, hl)
    for hl in (0, 1, 63):
        kl, _ = api._refine(1, "overlaps", l, r, None, A, B, heavy_log2=hl)
        assert set(kl.cpu().tolist()) == {2, 6}, hl
        kl, _ = api._refine(1, "contains_properly", r, l, None, B, A, heavy_log2=hl)
        assert set(kl.cpu().tolist()) == {4}, hl


@pytest.mark.parametrize("per_side", [1, 2, 5])
def test_rows_that_share_edges(per_side):
    """A grid of squares, each side in one edge or several, with itself and with
    the squares inset by a quarter: contacts without a crossing, equal rows,
    nested rows, by every route, against the grid positions."""
    import torch

    from vibespatial_amd import api

    m = 6

    def square(i, j, d):
        t = [k / per_side for k in range(per_side)]
        w = 1 - 2 * d
        x, y = i + d, j + d
        return Polygon([(x + w * a, y) for a in t] + [(x + w, y + w * a) for a in t]
                       + [(x + w - w * a, y + w) for a in t] + [(x, y + w - w * a) for a in t])

    cells = [(i, j) for i in range(m) for j in range(m)]
    A = PolygonArray.from_geometries([square(i, j, 0.0) for i, j in cells])
    inner = PolygonArray.from_geometries([square(i, j, 0.25) for i, j in cells])
    pairs = [(a, b) for a in range(m * m) for b in range(m * m)
             if max(abs(cells[a][0] - cells[b][0]), abs(cells[a][1] - cells[b][1])) <= 1]
    l = torch.tensor([p[0] for p in pairs], dtype=torch.int64, device="cuda")
    r = torch.tensor([p[1] for p in pairs], dtype=torch.int64, device="cuda")
    same, other = {p for p in pairs if p[0] == p[1]}, {p for p in pairs if p[0] != p[1]}
    with_itself = {"intersects": same | other, "touches": other, "overlaps": set(), "within": same, "covers": same,
                   "contains_properly": set()}
    with_inner = {"intersects": same, "touches": set(), "overlaps": set(), "within": set(), "covers": same,
                  "contains_properly": same}
    for B, expect in ((A, with_itself), (inner, with_inner)):
        for pred, want in expect.items():
            for hl in (0, 1, 63):
                print(f"shared edges {per_side} {pred} {hl}", flush=True)
                kl, kr = api._refine(1, pred, l, r, None, A, B, heavy_log2=hl)
                assert set(zip(kl.tolist(), kr.tolist())) == want, (pred, hl)
