"""The radix sort where its path changes: one block up to 4,096 pairs, fused
digit offsets up to 128 tiles, scanned ones above."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from vibespatial_amd import _lib
from vibespatial_amd.device import ptr, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 1023, 1024, 1025, 4095, 4096, 4097, 128 * 4096, 128 * 4096 + 1])
@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("bits", [(0, None), (3, 14), (5, 6)])
def test_stable_on_every_path(n, key_bytes, bits):
    rng = np.random.default_rng(n)
    b0, b1 = bits[0], bits[1] or 8 * key_bytes
    npt = np.uint64 if key_bytes == 8 else np.uint32
    keys = rng.integers(0, 2**63, n, dtype=np.uint64).astype(npt)
    keys[rng.integers(0, n, n // 3)] = keys[0]  # a run of one key
    tk = torch.from_numpy(keys.view(np.int64 if key_bytes == 8 else np.int32)).cuda()
    vals = torch.arange(n, dtype=torch.int32, device="cuda")
    L = _lib.lib()
    ws = torch.empty(L.vs_sort_workspace_bytes(n, key_bytes), dtype=torch.uint8, device="cuda")
    fn = L.vs_sort_pairs_u64 if key_bytes == 8 else L.vs_sort_pairs_u32
    _lib.check(fn(ptr(tk), ptr(vals), n, b0, b1, ptr(ws), ws.numel(), stream()), "sort")
    digit = (keys >> npt(b0)) & npt(2 ** (b1 - b0) - 1)
    order = np.argsort(digit, kind="stable")
    assert np.array_equal(vals.cpu().numpy(), order)
    assert np.array_equal(tk.cpu().numpy().view(npt), keys[order])
