"""The WKB row passes at the edges of a wave's 64 and 256 rows, of a tile's
1,024, of four tiles and of the prefix's 4,096 tiles: points alone, one polygonal row at a wave's first or last place,
a null or a tagged point among plain ones, mixed byte orders, and a record that
is 21 bytes long and no point, against the oracle."""

from __future__ import annotations

import struct

import numpy as np
import pytest

from oracle import wkb_ref as W
from vibespatial_amd.io import decode_wkb

pytestmark = pytest.mark.gpu

SQUARE = b"\x01" + struct.pack("<III", 3, 1, 4) + struct.pack("<8d", 0, 0, 1, 0, 0, 1, 0, 0)
TWO = b"\x01" + struct.pack("<II", 6, 2) + SQUARE + SQUARE
EMPTIES = b"\x01" + struct.pack("<III", 3, 3, 0) + struct.pack("<II", 0, 0)  # 21 bytes: three empty rings
TAGGED = b"\x01" + struct.pack("<IIdd", 0x20000001, 4326, 5.0, 6.0)


@pytest.mark.parametrize("odd", [None, SQUARE, TWO, EMPTIES, TAGGED, b""], ids=lambda r: "none" if r is None else len(r))
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 1023, 1024, 1025, 4095, 4096, 4097, 9000])
def test_waves(n, odd):
    print(f"wkb waves n {n} odd {None if odd is None else len(odd)}", flush=True)
    rng = np.random.default_rng(n)
    xy = rng.uniform(-1e3, 1e3, (n, 2))
    recs = [struct.pack("<BIdd", 1, 1, *v) if k % 3 else struct.pack(">BIdd", 0, 1, *v) for k, v in enumerate(xy)]
    if odd is not None:
        for k in {0, 63, 64, 255, 256, 1023, 1024, 4095, 4096, n - 1} & set(range(n)):
            recs[k] = odd
    payload = np.frombuffer(b"\xee" * 3 + b"".join(recs), np.uint8)
    offsets = np.concatenate([[0], np.cumsum([len(r) for r in recs])]) + 3
    ga, exp = decode_wkb(payload, offsets, None), W.decode_column(payload, offsets, None)
    if ga.points is not None:
        assert np.array_equal(ga.points.x, exp["point_x"]) and np.array_equal(ga.points.y, exp["point_y"])
        assert np.array_equal(ga.point_rows, exp["point_rows"])
    assert (0 if ga.points is None else len(ga.point_rows)) == len(exp["point_rows"])
    assert (0 if ga.polygons is None else len(ga.polygon_rows)) == len(exp["polygon_rows"])
    if ga.polygons is not None:
        assert np.array_equal(ga.polygon_rows, exp["polygon_rows"])
        for k in ("x", "y", "ring_offsets", "part_offsets", "geom_offsets"):
            assert np.array_equal(getattr(ga.polygons, k), exp[k]), k


@pytest.mark.parametrize("extra", [-1, 0, 1, 1500])
def test_more_tiles_than_one_round_of_the_prefix(extra):
    """4,096 tiles of points, a square as the last record of each round."""
    n = 4096 * 1024 + extra
    print(f"wkb tiles n {n}", flush=True)
    rng = np.random.default_rng(extra + 1)
    rec = np.zeros(n, dtype=np.dtype([("order", "u1"), ("type", "<u4"), ("x", "<f8"), ("y", "<f8")]))
    rec["order"], rec["type"] = 1, 1
    rec["x"], rec["y"] = rng.uniform(-1e3, 1e3, (2, n))
    at = sorted({4096 * 1024 - 1, n - 1} & set(range(n)))
    cuts = [0, *(k * 21 for k in at), n * 21]
    raw = rec.tobytes()
    payload = b"".join(raw[a + 21 * (i > 0) : b] + (SQUARE if i < len(at) else b"")
                       for i, (a, b) in enumerate(zip(cuts, cuts[1:])))
    size = np.full(n, 21, dtype=np.int64)
    size[at] = len(SQUARE)
    ga = decode_wkb(np.frombuffer(payload, np.uint8), np.concatenate([[0], np.cumsum(size)]), None)
    keep = np.ones(n, dtype=bool)
    keep[at] = False
    assert np.array_equal(ga.point_rows, np.flatnonzero(keep)) and np.array_equal(ga.polygon_rows, at)
    assert np.array_equal(ga.points.x, rec["x"][keep]) and np.array_equal(ga.points.y, rec["y"][keep])
    assert np.array_equal(ga.polygons.ring_offsets, 4 * np.arange(len(at) + 1))
