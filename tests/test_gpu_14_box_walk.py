"""Box queries of few hits per box: units of 64 and of 16 boxes, unions split
down to 4 boxes, every fanout's groups per step, the smallest trees, and its
stack at the fullest."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from vibespatial_amd import _lib
from vibespatial_amd import join as J

pytestmark = pytest.mark.gpu


def _boxes(rng, n, extent, side):
    c = rng.uniform(0, extent, (n, 2))
    h = rng.uniform(0, side, (n, 2)) / 2
    return np.column_stack([c - h, c + h])


@pytest.mark.parametrize("n_q,n_t,fanout", [(1, 1, 16), (15, 2, 2), (17, 16, 16), (65, 17, 16), (400, 1000, 2),
                                            (400, 1000, 3), (700, 5000, 16), (700, 5000, 64), (3000, 20_000, 16),
                                            (262_143, 300, 16), (262_144, 300, 16), (524_287, 300, 16),
                                            (524_290, 300, 16)])
def test_sparse_and_dense_queries_match_bruteforce(n_q, n_t, fanout):
    rng = np.random.default_rng(n_q + n_t)
    tb = _boxes(rng, n_t, 1000.0, 20.0)
    qb = _boxes(rng, n_q, 1000.0, 4.0)
    if n_q > 20:
        qb[: n_q // 3] = qb[0] + rng.normal(0, 1, (n_q // 3, 1))  # a dense patch beside the scattered boxes
        qb[rng.integers(1, n_q, 5)] = np.nan
        tb[rng.integers(1, n_t, 2)] = np.nan if n_t > 100 else tb[0]
    tree = J.build_tree(torch.from_numpy(tb).cuda(), fanout=fanout)
    el, er = [], []
    for t in range(n_t) if n_t < n_q else ():
        k = np.flatnonzero((qb[:, 0] <= tb[t, 2]) & (qb[:, 2] >= tb[t, 0]) & (qb[:, 1] <= tb[t, 3])
                           & (qb[:, 3] >= tb[t, 1]))
        el.append(k)
        er.append(np.full(len(k), t))
    for q in range(n_q) if n_t >= n_q else ():
        k = np.flatnonzero((qb[q, 0] <= tb[:, 2]) & (qb[q, 2] >= tb[:, 0]) & (qb[q, 1] <= tb[:, 3])
                           & (qb[q, 3] >= tb[:, 1]))
        el.append(np.full(len(k), q))
        er.append(k)
    el, er = np.concatenate(el), np.concatenate(er)
    o = np.lexsort((er, el))
    q = torch.from_numpy(qb).cuda()
    for cap in (31 * n_q, max(4, len(el) // 2)):  # below the one-box shape; and a retry
        l, r, st = J.query_boxes(q, tree, capacity=cap)
        assert np.array_equal(l.cpu().numpy(), el[o]) and np.array_equal(r.cpu().numpy(), er[o])


@pytest.mark.parametrize("n_t,fanout", [(32_768, 2), (177_147, 3), (262_144, 4), (100_000, 16), (300_000, 64)])
def test_boxes_over_whole_deep_trees(n_t, fanout):
    """Boxes that cover every item open every node: the walk's stack at its fullest."""
    print(f"box walk over {n_t} items, fanout {fanout}", flush=True)
    rng = np.random.default_rng(fanout)
    tb = _boxes(rng, n_t, 1000.0, 1.0)
    qb = np.tile([-1e4, -1e4, 1e4, 1e4], (18, 1))  # one unit of 16 boxes and one of 2
    qb[3], qb[11] = [500.0, 500.0, 520.0, 520.0], np.nan
    tree = J.build_tree(torch.from_numpy(tb).cuda(), fanout=fanout)
    hit = (qb[:, None, 0] <= tb[:, 2]) & (qb[:, None, 2] >= tb[:, 0]) & (qb[:, None, 1] <= tb[:, 3]) & \
        (qb[:, None, 3] >= tb[:, 1])
    el, er = np.nonzero(hit)
    # the walk counts every pair into too few slots, then the other shape writes them
    l, r, st = J.query_boxes(torch.from_numpy(qb).cuda(), tree, capacity=31 * 18)
    assert st.retries == 1 and st.staged == len(el)
    assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er)


def test_layout_too_deep_for_the_walk_takes_the_other_shape():
    """16 levels of fanout 32, 619 nodes staged: more entries than the walk's
    stack is sized for; the pairs are those of a plain search."""
    print("box walk, layout too deep", flush=True)
    rng = np.random.default_rng(5)
    counts = [1, 20, 619] + [700] * 13
    tb = _boxes(rng, 700, 1000.0, 30.0)
    qb = _boxes(rng, 90, 1000.0, 60.0)
    layout = _lib.TreeLayout(fanout=32, n_levels=16, n_items=700, n_nodes=sum(counts))
    boxes = []
    for k, c in enumerate(counts):
        layout.level_start[k] = sum(counts[:k])
        layout.level_count[k] = c
        b = np.full((c, 4), np.nan)
        below = counts[k + 1] if k < 15 else 0
        b[: -(-below // 32)] = [-100.0, -100.0, 1100.0, 1100.0]  # the nodes that have children
        boxes.append(tb if k == 15 else b)
    dev = torch.device("cuda")
    tree = J.DeviceTree(layout, torch.from_numpy(np.concatenate(boxes)).to(dev),
                        torch.arange(700, dtype=torch.int32, device=dev), None, None)
    hit = (qb[:, None, 0] <= tb[:, 2]) & (qb[:, None, 2] >= tb[:, 0]) & (qb[:, None, 1] <= tb[:, 3]) & \
        (qb[:, None, 3] >= tb[:, 1])
    el, er = np.nonzero(hit)
    l, r, _ = J.query_boxes(torch.from_numpy(qb).to(dev), tree, capacity=31 * 90)
    assert np.array_equal(l.cpu().numpy(), el) and np.array_equal(r.cpu().numpy(), er) and len(el) < 31 * 90
