"""Batched joins at the limits of the job keys (32 bits up to 65,536 jobs) and
with one job whose tree is deep and whose left rows are scattered, and rings of
one coordinate, the last of them at the end of the coordinate buffer."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from vibespatial_amd import join as J
from vibespatial_amd import synthetic as S
from vibespatial_amd.device import DevicePolygons
from vibespatial_amd.geometry import PolygonArray

pytestmark = pytest.mark.gpu


def _stars(rng, n, extent, r):
    return S.star_polygons(rng, rng.uniform(0, extent, n), rng.uniform(0, extent, n), rng.uniform(r / 2, r, n),
                           rng.integers(4, 13, n))


@pytest.mark.parametrize("n_jobs,per_left,per_right", [(1, 300, 1), (1, 700, 20_000), (3, 4_000, 17), (65_536, 1, 1),
                                                       (65_537, 1, 1), (70_000, 2, 1)])
def test_pairs_of_every_job_match_oracle(n_jobs, per_left, per_right):
    rng = np.random.default_rng(n_jobs + per_right)
    extent = 10.0 if per_right == 1 else 500.0  # one right row a job: packed so that some pairs meet
    A, B = _stars(rng, n_jobs * per_left, extent, 5.0), _stars(rng, n_jobs * per_right, extent, 6.0)
    lj, rj = (torch.arange(n_jobs + 1, dtype=torch.int64, device="cuda") * k for k in (per_left, per_right))
    l, r, _ = J.batched_intersects(DevicePolygons.from_host(A), DevicePolygons.from_host(B), lj, rj)
    l, r = l.cpu().numpy(), r.cpu().numpy()
    if n_jobs <= 100:
        el, er = oracle.sjoin_polygons_polygons(A, B)
        keep = el // per_left == er // per_right
        el, er = el[keep], er[keep]
    else:
        el = np.arange(n_jobs * per_left)
        er = el // per_left  # one right row a job
        keep = np.array([oracle.polygon_intersects(A, int(a), B, int(b)) for a, b in zip(el, er)])
        el, er = el[keep], er[keep]
    assert np.array_equal(l, el) and np.array_equal(r, er) and len(l) > 0


def _single_rings(rings):
    n = len(rings)
    xy = np.concatenate([np.asarray(r, dtype=np.float64).reshape(-1, 2) for r in rings])
    rows = np.arange(n + 1, dtype=np.int32)
    return PolygonArray(xy[:, 0].copy(), xy[:, 1].copy(), np.cumsum([0] + [len(r) for r in rings]).astype(np.int32),
                        rows, rows)


@pytest.mark.parametrize("cell_grid", [True, False])
def test_rings_of_one_coordinate(cell_grid):
    print(f"one-coordinate rings, cell grid {cell_grid}", flush=True)
    square = [(0, 0), (4, 0), (4, 4), (0, 4), (0, 0)]
    A = _single_rings([square, [(2, 2)], [(4, 4)], [(0, 2)], [(9, 9)], [(7, 7)]])
    B = _single_rings([[(7, 7)], square, [(2, 2)], [(0, 2)], [(9, 9)], [(4, 4)]])
    offsets = torch.tensor([0, 6], dtype=torch.int64, device="cuda")
    l, r, _ = J.batched_intersects(DevicePolygons.from_host(A), DevicePolygons.from_host(B), offsets, offsets,
                                   cell_grid=cell_grid)
    el, er = oracle.sjoin_polygons_polygons(A, B)
    assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er) and len(el) > 0
