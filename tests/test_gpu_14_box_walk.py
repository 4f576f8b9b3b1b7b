"""Box queries of few hits per box: units of 64 and of 16 boxes, unions split
down to 4 boxes, every fanout's groups per step, the smallest trees."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from vibespatial_amd import join as J

pytestmark = pytest.mark.gpu


def _boxes(rng, n, extent, side):
    c = rng.uniform(0, extent, (n, 2))
    h = rng.uniform(0, side, (n, 2)) / 2
    return np.column_stack([c - h, c + h])


@pytest.mark.parametrize("n_q,n_t,fanout", [(1, 1, 16), (15, 2, 2), (17, 16, 16), (65, 17, 16), (400, 1000, 2),
                                            (400, 1000, 3), (700, 5000, 16), (700, 5000, 64), (3000, 20_000, 16),
                                            (524_287, 300, 16), (524_290, 300, 16)])
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
