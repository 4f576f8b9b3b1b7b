"""The finish pass that sorts by both ids, on either side of the capacity from
which it is used (32 slots per left row, 16 known pairs) and around the radix digit edges."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from vibespatial_amd import join as J
from vibespatial_amd.device import DevicePoints

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_left,n_right", [(2, 3), (3, 256), (256, 257), (257, 65_536), (300, 65_537), (1000, 70_001)])
def test_both_finishes_give_the_lexsorted_pairs(n_left, n_right):
    rng = np.random.default_rng(n_left + n_right)
    x, y = rng.uniform(0, 1, n_right), rng.uniform(0, 1, n_right)
    half = 0.5 * np.sqrt(20.0 / n_right)
    cx, cy = rng.uniform(0, 1, n_left), rng.uniform(0, 1, n_left)
    boxes = np.column_stack([cx - half, cy - half, cx + half, cy + half])
    inside = (x >= boxes[:, :1]) & (x <= boxes[:, 2:3]) & (y >= boxes[:, 1:2]) & (y <= boxes[:, 3:4])
    el, er = np.nonzero(inside)
    Q = DevicePoints(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    qb = torch.from_numpy(boxes).cuda()
    tree = J.build_tree(J.point_boxes(Q))
    idx = J.LearnedPointIndex(Q)
    for slots in (31 * n_left, 32 * n_left - 1, 32 * n_left, 40 * n_left + 4096):
        for got in (J.query_boxes(qb, tree, capacity=slots), idx.query_boxes(qb, capacity=slots)):
            assert np.array_equal(got[0].cpu().numpy(), el) and np.array_equal(got[1].cpu().numpy(), er), slots


@pytest.mark.parametrize("n_left,n_right", [(2, 3), (256, 257), (257, 65_536), (1000, 70_001)])
@pytest.mark.parametrize("hits", [5, 15, 17])
def test_the_line_between_the_finishes(n_left, n_right, hits):
    """Even rows with one of a hundred pairs among them, below the line (16
    known pairs a row, 32 slots of a given capacity) as above it."""
    rng = np.random.default_rng(n_left + n_right)
    x, y = rng.uniform(0, 1, n_right), rng.uniform(0, 1, n_right)
    half = np.full(n_left, 0.5 * np.sqrt(hits / n_right))
    half[-1] = 0.5 * np.sqrt(100.0 / n_right)
    cx, cy = rng.uniform(0.1, 0.9, n_left), rng.uniform(0.1, 0.9, n_left)
    boxes = np.column_stack([cx - half, cy - half, cx + half, cy + half])
    inside = (x >= boxes[:, :1]) & (x <= boxes[:, 2:3]) & (y >= boxes[:, 1:2]) & (y <= boxes[:, 3:4])
    el, er = np.nonzero(inside)
    Q = DevicePoints(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    qb = torch.from_numpy(boxes).cuda()
    tree = J.build_tree(J.point_boxes(Q))
    idx = J.LearnedPointIndex(Q)
    got = [idx.query_boxes(qb)]  # the pairs are counted first
    for slots in (32 * n_left - 1, 32 * n_left):
        got += [J.query_boxes(qb, tree, capacity=slots), idx.query_boxes(qb, capacity=slots)]
    for l, r, _ in got:
        assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er)
