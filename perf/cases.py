"""The calls whose time is measured: what a program does with this package, from
one small query to the sizes of its benchmark, through the public entry points.

Kinds:
  join      GeoSeries(polygons).sindex.query(points, predicate): the point x
            polygon spatial join, the index over the polygons kept
  boxes     a new SpatialIndex over a point column, queried once by
            rectangles: the index build and the box query in one pass
  contains  polygons over a point column whose index is kept
  relate    polygon x polygon predicates through sindex.query
  batched   many independent polygon x polygon intersects joins in one call
  dwithin   sindex.query(predicate="dwithin"), one or one-per-row distances
  nearest   sindex.nearest with distances, on host arrays
  wkb       decoding a WKB column that is in device memory

Inputs are drawn on the GPU.  Points follow a Gaussian mixture (or are uniform,
or sit in Zipf-weighted clusters), polygons are star polygons with log-normal
vertex counts, holes and, where asked, second parts.  Extents grow with the
number of polygons, so a point meets about as many polygons at every size as in
the benchmark's 10M x 100k join.

The number of matching pairs is part of an answer's shape, so a case always has
the same map: the case draws its layout, and the seed draws the order of its
rows (points and polygons alike come in random order) and which way the map is
turned and mirrored.  Both keep every relation exactly as it was and change
every buffer, every key order and every row number of the answer.
"""

from __future__ import annotations

import math
import zlib

import torch

from vibespatial_amd import join as J
from vibespatial_amd.api import GeoSeries, SpatialIndex
from vibespatial_amd.device import DevicePoints, DevicePolygons, device_points, device_polygons
from vibespatial_amd.geometry import PointArray, PolygonArray, as_geometry_array, box_array
from vibespatial_amd.io import decode_wkb_device

DEVICE = torch.device("cuda")
F64 = torch.float64
UTM = (5.0e5, 3.0e6)  # easting / northing of data in projected coordinates


def listed():
    return [
        # one small lookup inside a program's loop: a thousand points against
        # a few dozen zones, the answer as host arrays; launches and latency
        dict(name="join_1k", kind="join", points=1003, polygons=57, predicate="within", cloud="uniform", utm=False,
             multi=0.0, host=True),
        # a city's worth of points against its districts, host arrays back
        dict(name="join_100k", kind="join", points=100_000, polygons=1_000, predicate="within", cloud="uniform",
             utm=False, multi=0.0, host=True),
        # points on shared boundaries in projected coordinates, some rows of
        # two parts: the exact path is taken often
        dict(name="join_utm_1m", kind="join", points=1_000_003, polygons=100_003, predicate="intersects", cloud="gmm",
             utm=True, multi=0.05, host=False),
        # the benchmark's join
        dict(name="join_10m", kind="join", points=10_000_000, polygons=100_000, predicate="within", cloud="gmm",
             utm=False, multi=0.0, host=False),
        # window queries over a point table loaded once: build and query
        dict(name="boxes_10m", kind="boxes", points=10_000_001, boxes=50_000),
        # zones asking which of the indexed points they hold
        dict(name="contains_5m", kind="contains", points=5_000_011, polygons=20_000, predicate="contains", multi=0.02),
        # two small polygon layers
        dict(name="relate_2k", kind="relate", left=2_003, right=1_999, predicate="intersects", multi=0.0),
        # two large polygon layers, a relation that needs the full test
        dict(name="relate_100k", kind="relate", left=100_000, right=100_000, predicate="overlaps", multi=0.0),
        # building footprints against parcels, one job per map tile
        dict(name="batched_4096", kind="batched", jobs=4096),
        # everything within 25 m of a zone
        dict(name="dwithin_3m", kind="dwithin", points=3_000_017, polygons=100_000, distance=25.0, per_row=False),
        # the closest zone of every point, with its distance
        dict(name="nearest_1m", kind="nearest", points=1_000_003, polygons=100_000),
        # reading a GeoParquet geometry column
        dict(name="wkb_10m", kind="wkb", points=10_000_000, polygons=100_000, multi=0.0, little=True, shuffled=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) | 1


def draw(rng):
    kind = rng.choice(("join", "join", "boxes", "contains", "relate", "batched", "dwithin", "nearest", "wkb"))
    if kind == "join":
        n = _log_int(rng, 500, 9_999_999)
        utm = rng.random() < 0.4  # only there do points sit on boundaries
        return dict(kind=kind, points=n, polygons=_log_int(rng, 20, 99_999),
                    predicate=rng.choice(("within", "intersects", "covered_by") + ("touches",) * utm),
                    cloud=rng.choice(("uniform", "gmm")), utm=utm, multi=rng.choice((0.0, 0.05)), host=n <= 200_000)
    if kind == "boxes":
        n = _log_int(rng, 5_000, 9_999_999)
        return dict(kind=kind, points=n, boxes=_log_int(rng, 50, 49_999))
    if kind == "contains":
        return dict(kind=kind, points=_log_int(rng, 5_000, 4_999_999), polygons=_log_int(rng, 10, 19_999),
                    predicate=rng.choice(("contains", "covers", "intersects")), multi=rng.choice((0.0, 0.02)))
    if kind == "relate":
        return dict(kind=kind, left=_log_int(rng, 1_000, 99_999), right=_log_int(rng, 1_000, 99_999),
                    predicate=rng.choice(("intersects", "overlaps", "within", "contains")),
                    multi=rng.choice((0.0, 0.02)))
    if kind == "batched":
        return dict(kind=kind, jobs=_log_int(rng, 2, 4095))
    if kind == "dwithin":
        return dict(kind=kind, points=_log_int(rng, 500, 2_999_999), polygons=_log_int(rng, 20, 99_999),
                    distance=rng.choice((1.0, 10.0, 25.0)), per_row=rng.random() < 0.3)
    if kind == "nearest":
        return dict(kind=kind, points=_log_int(rng, 500, 999_999), polygons=_log_int(rng, 50, 99_999))
    return dict(kind=kind, points=_log_int(rng, 100, 9_999_999), polygons=_log_int(rng, 10, 99_999),
                multi=rng.choice((0.0, 0.1)), little=rng.random() < 0.7, shuffled=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Draws:
    """Random numbers on the device, from one seed."""

    @classmethod
    def layout(cls, case):
        """The draws of a case's map: the same for every seed."""
        text = repr(sorted((k, v) for k, v in case.items() if k not in ("name", "host", "predicate", "little")))
        return cls(zlib.crc32(text.encode()))

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(int(seed) & (2**62 - 1))

    def u(self, n, lo=0.0, hi=1.0):
        return torch.rand(n, generator=self.g, device=DEVICE, dtype=F64) * (hi - lo) + lo

    def normal(self, n):
        return torch.randn(n, generator=self.g, device=DEVICE, dtype=F64)

    def ints(self, n, lo, hi):
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEVICE)

    def order(self, n):
        return torch.argsort(self.u(n))

    def lognormal(self, n, median, sigma, lo, hi):
        return torch.exp(math.log(median) + sigma * self.normal(n)).round().clamp(lo, hi).long()


def _starts(counts):
    """Exclusive prefix sums with the total behind them."""
    out = torch.zeros(counts.numel() + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(counts, 0, out=out[1:])
    return out


def _rows_of(starts):
    """The row of every entry of rows that begin at `starts`."""
    n = starts.numel() - 1
    return torch.repeat_interleave(torch.arange(n, device=DEVICE), starts[1:] - starts[:-1])


def _stars(d, cx, cy, radius, vertices, holes=None, multi=0.0):
    """Star polygons as (x, y, ring, part, geom offsets).  Vertex k of n sits in
    the k-th of n equal sectors, so no edge spans half a turn and every ring is
    simple.  `holes` (0 to 3 per polygon) lie inside 0.9 of the shell's
    inscribed circle, one in the middle or several side by side; a share
    `multi` of the rows gets a second part beside the first."""
    m = cx.numel()
    n_parts = torch.ones(m, dtype=torch.int64, device=DEVICE)
    if multi:
        n_parts += (d.u(m) < multi).long()
    geom = _starts(n_parts)
    row = _rows_of(geom)
    parts = row.numel()
    second = torch.arange(parts, device=DEVICE) - geom[row]  # 0 or 1
    pcx, pcy = cx[row] + 2.7 * radius[row] * second, cy[row]
    prad = radius[row]
    pholes = torch.zeros(parts, dtype=torch.int64, device=DEVICE) if holes is None else holes[row]
    part = _starts(pholes + 1)
    ring_part = _rows_of(part)
    rings = ring_part.numel()
    which = torch.arange(rings, device=DEVICE) - part[ring_part]  # 0: the shell
    shell = which == 0
    n = torch.where(shell, vertices[row][ring_part], d.ints(rings, 4, 17))
    ring = _starts(n + 1)
    rr = _rows_of(ring)
    total = rr.numel()
    local = torch.arange(total, device=DEVICE) - ring[rr]
    local = torch.where(local == n[rr], torch.zeros_like(local), local)  # a ring closes on its first vertex
    local = torch.where(shell[rr], local, n[rr] - 1 - local)  # holes run clockwise
    at = ring[rr] + local
    ang = (local + d.u(total, 0.05, 0.95)[at]) * (2 * math.pi) / n[rr]
    rad = 1.0 + d.u(total, -0.3, 0.3)[at]
    ux, uy = rad * torch.cos(ang), rad * torch.sin(ang)
    rx, ry = pcx[ring_part], pcy[ring_part]
    rscale = prad[ring_part]
    if holes is not None:
        # inscribed radius of every ring at scale 1: the least distance of its
        # edges from the centre
        ex, ey = torch.roll(ux, -1) - ux, torch.roll(uy, -1) - uy
        t = (-(ux * ex + uy * ey) / (ex * ex + ey * ey)).clamp(0.0, 1.0)
        dist = torch.hypot(ux + t * ex, uy + t * ey)
        dist[ring[1:] - 1] = float("inf")  # no edge leaves a closing vertex
        inner = torch.full((rings,), float("inf"), dtype=F64, device=DEVICE)
        inner.scatter_reduce_(0, rr, dist, "amin")
        inner = inner[part[:-1]][ring_part] * prad[ring_part]
        k = pholes[ring_part]
        alone = k == 1
        off = torch.where(alone, torch.zeros_like(inner), 0.5 * inner)
        room = torch.where(alone, inner, torch.minimum(0.5 * inner, off * torch.sin(math.pi / k.clamp(min=1))))
        size = torch.minimum(d.u(rings, 0.1, 0.4) * prad[ring_part], 0.9 / 1.3 * room)
        turn = d.u(parts, 0.0, 2 * math.pi)[ring_part] + 2 * math.pi * (which - 1) / k.clamp(min=1)
        rscale = torch.where(shell, rscale, size)
        rx = torch.where(shell, rx, rx + off * torch.cos(turn))
        ry = torch.where(shell, ry, ry + off * torch.sin(turn))
    x, y = rx[rr] + rscale[rr] * ux, ry[rr] + rscale[rr] * uy
    return x, y, ring.int(), part.int(), geom.int()


def _take(s, rows):
    """The polygons `rows` of s, in that order."""
    x, y, ring, part, geom = s[0], s[1], s[2].long(), s[3].long(), s[4].long()
    at = rows
    out = []
    for off in (geom, part, ring):
        first = _starts(off[at + 1] - off[at])
        k = _rows_of(first)
        at = off[at][k] + torch.arange(k.numel(), device=DEVICE) - first[k]
        out.append(first.int())
    return x[at], y[at], out[2], out[1], out[0]


class _Turn:
    """One of the eight turns and mirrorings of the plane that are exact in
    floating point."""

    def __init__(self, d):
        self.swap, self.neg_x, self.neg_y = (d.u(3) < 0.5).tolist()

    def __call__(self, x, y):
        if self.swap:
            x, y = y, x
        return (-x if self.neg_x else x), (-y if self.neg_y else y)

    def polygons(self, s):
        return (*self(s[0], s[1]), *s[2:])

    def boxes(self, b):
        x0, y0 = self(b[:, 0], b[:, 1])
        x1, y1 = self(b[:, 2], b[:, 3])
        return torch.stack([torch.minimum(x0, x1), torch.minimum(y0, y1), torch.maximum(x0, x1),
                            torch.maximum(y0, y1)], 1)


def _extent(polygons):
    """Side of the square that `polygons` zones of the benchmark's sizes fill as
    densely as 100,000 of them fill 1e5 x 1e5."""
    return 1e5 * math.sqrt(polygons / 1e5)


def _zones(d, m, extent, shift=(0.0, 0.0), multi=0.0):
    return _stars(d, shift[0] + d.u(m, 0.0, extent), shift[1] + d.u(m, 0.0, extent), d.u(m, 50.0, 300.0),
                  d.lognormal(m, 24.0, 1.0, 4, 10_000), d.ints(m, 0, 4), multi)


def _cloud(d, n, extent, cloud="gmm", shift=(0.0, 0.0)):
    if cloud == "uniform":
        return shift[0] + d.u(n, 0.0, extent), shift[1] + d.u(n, 0.0, extent)
    mx, my, sg = d.u(64, 0.0, extent), d.u(64, 0.0, extent), d.u(64, 0.002, 0.03) * extent
    c = d.ints(n, 0, 64)
    return shift[0] + mx[c] + sg[c] * d.normal(n), shift[1] + my[c] + sg[c] * d.normal(n)


def _host_points(x, y):
    pa = PointArray(x.cpu().numpy(), y.cpu().numpy())
    device_points(pa)
    as_geometry_array(pa)
    return pa


def _host_polygons(s):
    pa = PolygonArray(*(t.cpu().numpy() for t in s))
    device_polygons(pa)
    as_geometry_array(pa)
    return pa


def _join_inputs(case, seed):
    """(x, y, polygons, distance per point or None) of a case and seed."""
    d = _Draws.layout(case)
    shift = UTM if case.get("utm") else (0.0, 0.0)
    extent = _extent(case["polygons"])
    s = _zones(d, case["polygons"], extent, shift, case.get("multi", 0.0))
    x, y = _cloud(d, case["points"], extent, case.get("cloud", "gmm"), shift)
    if case.get("utm"):  # one point in twenty sits on a vertex
        k = max(1, case["points"] // 20)
        at, v = d.order(case["points"])[:k], d.ints(k, 0, s[0].numel())
        x[at], y[at] = s[0][v], s[1][v]
    dist = d.u(case["points"], 0.0, case["distance"]) if case.get("per_row") else None
    d = _Draws(seed)
    turn, order = _Turn(d), d.order(case["points"])
    x, y = turn(x[order], y[order])
    return x, y, turn.polygons(_take(s, d.order(case["polygons"]))), None if dist is None else dist[order]


def _relate_inputs(case, seed):
    d, e = _Draws.layout(case), _Draws(seed)
    extent, turn = _extent(max(case["left"], case["right"])), _Turn(e)
    sides = [_zones(d, case[k], extent, multi=case["multi"]) for k in ("left", "right")]
    return [turn.polygons(_take(s, e.order(s[4].numel() - 1))) for s in sides]


def _zipf(d, n, w, cx, cy):
    c = torch.searchsorted(w, d.u(n)).clamp(max=w.numel() - 1)
    return cx[c] + 500.0 * d.normal(n), cy[c] + 500.0 * d.normal(n)


def _box_inputs(case, seed):
    d = _Draws.layout(case)
    w = 1.0 / torch.arange(1, 1025, dtype=F64, device=DEVICE) ** 1.1
    w = torch.cumsum(w / w.sum(), 0)
    cx, cy = d.u(1024, 0.0, 1e5), d.u(1024, 0.0, 1e5)
    x, y = _zipf(d, case["points"], w, cx, cy)
    bx, by = _zipf(d, case["boxes"], w, cx, cy)
    bw = torch.exp(math.log(50.0) + d.normal(case["boxes"])) / 2
    bh = torch.exp(math.log(50.0) + d.normal(case["boxes"])) / 2
    boxes = torch.stack([bx - bw, by - bh, bx + bw, by + bh], 1)
    d = _Draws(seed)
    turn, order = _Turn(d), d.order(case["points"])
    return (*turn(x[order], y[order]), turn.boxes(boxes[d.order(case["boxes"])]))


def _batch_inputs(case, seed):
    """(polygons, first row of every job) of both sides; the seed draws the
    order of the jobs and of the rows of each job."""
    d, e = _Draws.layout(case), _Draws(seed)
    jobs = case["jobs"]
    turn, place = _Turn(e), e.order(jobs)
    nl = d.lognormal(jobs, 2000.0, 1.0, 1_000, 200_000)
    nr = d.lognormal(jobs, 300.0, 1.0, 10, 5_000)
    side = 120.0 * nr.to(F64).sqrt()
    j = torch.arange(jobs, device=DEVICE)
    ox, oy = (j % 64) * 2.0e4, torch.div(j, 64, rounding_mode="floor") * 2.0e4
    out = []
    for rows, lo, hi in ((nl, 2.5, 20.0), (nr, 40.0, 70.0)):
        start = _starts(rows)
        k = _rows_of(start)
        m = k.numel()
        nv = d.ints(m, 4, 13) if lo < 40.0 else d.lognormal(m, 40.0, 0.5, 4, 400)
        s = _stars(d, ox[k] + d.u(m) * side[k], oy[k] + d.u(m) * side[k], d.u(m, lo, hi), nv)
        order = torch.argsort(place[k] + e.u(m, 0.0, 0.999))
        ordered = torch.empty_like(rows)
        ordered[place] = rows
        out += [turn.polygons(_take(s, order)), _starts(ordered)]
    return out


def _put(payload, at, values, little):
    """Bytes of `values` (one number each) into payload from `at` on."""
    b = values.contiguous().view(torch.uint8).view(values.numel(), values.element_size())
    if not little:
        b = b.flip(1)
    payload[at[:, None] + torch.arange(b.shape[1], device=DEVICE)] = b


def _encode(x, y, s, little, order):
    """WKB column (payload, offsets) of the points and polygons; record k of
    `order` is a point (below the number of points) or a polygon."""
    px, py, ring, part, geom = s[0], s[1], s[2].long(), s[3].long(), s[4].long()
    n, m = x.numel(), geom.numel() - 1
    n_parts = geom[1:] - geom[:-1]
    c0 = ring[part[geom]]
    r0 = part[geom]
    several = n_parts > 1
    size = 9 + 4 * (r0[1:] - r0[:-1]) + 16 * (c0[1:] - c0[:-1]) + torch.where(several, 9 * n_parts, 0)
    length = torch.cat([torch.full((n,), 21, dtype=torch.int64, device=DEVICE), size])
    offsets = _starts(length[order])
    begin = torch.empty(n + m, dtype=torch.int64, device=DEVICE)
    begin[order] = offsets[:-1]
    payload = torch.zeros(int(offsets[-1]), dtype=torch.uint8, device=DEVICE)

    def head(at, kind, count=None):
        payload[at] = 1 if little else 0
        _put(payload, at + 1, kind.int(), little)
        if count is not None:
            _put(payload, at + 5, count.int(), little)

    pts, rows = begin[:n], begin[n:]
    if n:
        head(pts, torch.ones(n, device=DEVICE))
        _put(payload, pts + 5, x, little)
        _put(payload, pts + 13, y, little)
    # a row of one part is a Polygon record, one of several a MultiPolygon of them
    head(rows[several], torch.full((int(several.sum()),), 6, device=DEVICE), n_parts[several])
    g = _rows_of(geom)
    p = torch.arange(g.numel(), device=DEVICE)
    part_at = rows[g] + torch.where(several[g], 9 * (p - geom[g] + 1), 0) \
        + 4 * (part[p] - r0[g]) + 16 * (ring[part[p]] - c0[g])
    head(part_at, torch.full((g.numel(),), 3, device=DEVICE), part[1:] - part[:-1])
    rp = _rows_of(part)
    r = torch.arange(rp.numel(), device=DEVICE)
    ring_at = part_at[rp] + 9 + 4 * (r - part[rp]) + 16 * (ring[r] - ring[part[rp]])
    _put(payload, ring_at, (ring[1:] - ring[:-1]).int(), little)
    cr = _rows_of(ring)
    at = ring_at[cr] + 4 + 16 * (torch.arange(cr.numel(), device=DEVICE) - ring[cr])
    _put(payload, at, px, little)
    _put(payload, at + 8, py, little)
    return payload, offsets


def _wkb_inputs(case, seed):
    d = _Draws.layout(case)
    extent = _extent(case["polygons"])
    s = _zones(d, case["polygons"], extent, multi=case["multi"])
    x, y = _cloud(d, case["points"], extent)
    d = _Draws(seed)
    turn, order = _Turn(d), d.order(case["points"])
    x, y = turn(x[order], y[order])
    s = turn.polygons(_take(s, d.order(case["polygons"])))
    rows = case["points"] + case["polygons"]
    return x, y, s, d.order(rows) if case["shuffled"] else torch.arange(rows, device=DEVICE)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("join", "dwithin", "nearest", "contains"):
        x, y, s, dist = _join_inputs(case, seed)
        points, zones = _host_points(x, y), _host_polygons(s)
        if kind == "contains":
            index = GeoSeries(points).sindex
            index.query(zones, predicate="contains", return_device=True)  # the kept index
            return dict(kind=kind, index=index, query=zones, predicate=case["predicate"])
        state = dict(kind=kind, index=GeoSeries(zones).sindex, query=points)
        if kind == "join":
            state.update(predicate=case["predicate"], device=not case["host"])
        elif kind == "dwithin":
            state.update(distance=case["distance"] if dist is None else dist.cpu().numpy())
        return state
    if kind == "boxes":
        x, y, boxes = _box_inputs(case, seed)
        return dict(kind=kind, points=_host_points(x, y), query=_host_rectangles(boxes))
    if kind == "relate":
        a, b = (_host_polygons(s) for s in _relate_inputs(case, seed))
        return dict(kind=kind, index=GeoSeries(b).sindex, query=a, predicate=case["predicate"])
    if kind == "batched":
        a, lj, b, rj = _batch_inputs(case, seed)
        return dict(kind=kind, left=DevicePolygons(*a), right=DevicePolygons(*b), left_job=lj, right_job=rj)
    x, y, s, order = _wkb_inputs(case, seed)
    payload, offsets = _encode(x, y, s, case["little"], order)
    return dict(kind=kind, payload=payload, offsets=offsets,
                validity=torch.ones(offsets.numel() - 1, dtype=torch.uint8, device=DEVICE))


def _host_rectangles(boxes):
    pa = box_array(boxes.cpu().numpy())
    device_polygons(pa)
    as_geometry_array(pa)
    return pa


def run(state):
    kind = state["kind"]
    if kind == "join":
        return state["index"].query(state["query"], predicate=state["predicate"], return_device=state["device"])
    if kind == "boxes":
        return SpatialIndex(state["points"]).query(state["query"], predicate="intersects", return_device=True)
    if kind in ("contains", "relate"):
        return state["index"].query(state["query"], predicate=state["predicate"], return_device=True)
    if kind == "batched":
        left, right, _ = J.batched_intersects(state["left"], state["right"], state["left_job"], state["right_job"])
        return left, right
    if kind == "dwithin":
        return state["index"].query(state["query"], predicate="dwithin", distance=state["distance"],
                                    return_device=True)
    if kind == "nearest":
        pairs, distance = state["index"].nearest(state["query"], return_distance=True)
        return pairs, distance
    col = decode_wkb_device(state["payload"], state["offsets"], state["validity"])
    g = col.polygons
    return (col.points.x, col.points.y, col.point_rows, g.x, g.y, g.ring_offsets, g.part_offsets, g.geom_offsets,
            col.polygon_rows)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# Mean coordinates (16 B each) and rings (4 B each) of a zone, counting the
# closing vertices: a log-normal shell of mean 24 exp(1/2), 1.5 holes of 10.
ZONE = 16 * (24 * math.exp(0.5) + 1 + 1.5 * 11) + 4 * 2.5 + 8
PAIR = 16  # two int64 row numbers


def work(case):
    """Bytes: every input buffer read once and every output written once (the
    number of pairs is the expected one)."""
    kind = case["kind"]
    n, m = case.get("points", 0), case.get("polygons", 0)
    if kind in ("join", "contains"):
        pairs = (0.05 if case["predicate"] == "touches" else 0.9) * n
        return dict(bytes=16 * n + ZONE * m + PAIR * pairs, flops=0)
    if kind == "boxes":
        return dict(bytes=16 * n + (80 + 12) * case["boxes"] + PAIR * 1.02e-4 * n * case["boxes"], flops=0)
    if kind == "relate":
        a, b = case["left"], case["right"]
        pairs = (3.0 if case["predicate"] in ("intersects", "overlaps") else 0.1) * min(a, b)
        return dict(bytes=ZONE * (a + b) + PAIR * pairs, flops=0)
    if kind == "batched":
        left, right = 3500 * case["jobs"], 480 * case["jobs"]
        return dict(bytes=(16 * 9 + 12) * left + (16 * 46 + 12) * right + PAIR * left, flops=0)
    if kind == "dwithin":
        return dict(bytes=16 * n + ZONE * m + (8 * n if case["per_row"] else 8) + PAIR * 1.2 * n, flops=0)
    if kind == "nearest":
        return dict(bytes=16 * n + ZONE * m + (PAIR + 8) * 1.3 * n, flops=0)
    record = 9 * (n + m) + 8 * (n + m)  # offsets and validity in, row numbers out
    return dict(bytes=record + (21 + 16) * n + (9 + 2 * ZONE) * m, flops=0)


def tolerance(case):
    """Row numbers and copied coordinates are exact.  A distance is one fp64
    square root after a few fp64 operations on coordinates of up to 1e5, whose
    differences are exact or rounded once: 1e-13 covers another order of them."""
    return {"rel": 1e-13, "max": 1e-9, "differ": 0.0} if case["kind"] == "nearest" else "exact"


def exact(case, seed):
    """The computed numbers: decoded coordinates, and nearest distances by
    brute force where that is quick.  Row numbers have no 64-bit counterpart."""
    if case["kind"] == "wkb":
        x, y, s, order = _wkb_inputs(case, seed)
        n = case["points"]
        pts, rows = order[order < n], order[order >= n] - n
        # coordinates of the polygons in record order
        c = s[2].long()[s[3].long()[s[4].long()]]
        count = (c[1:] - c[:-1])[rows]
        first = _starts(count)
        k = _rows_of(first)
        at = c[rows][k] + torch.arange(k.numel(), device=DEVICE) - first[k]
        return (x[pts], y[pts], None, s[0][at], s[1][at], None, None, None, None)
    if case["kind"] == "nearest":
        x, y, s, _ = _join_inputs(case, seed)
        if x.numel() * s[0].numel() > 1e9:
            return None
        return (None, _nearest_distances(x, y, s))
    return None


def _nearest_distances(x, y, s):
    """Distance of every nearest (point, polygon) pair, in (point, polygon)
    order: all edges against chunks of points."""
    ring, part, geom = s[2].long(), s[3].long(), s[4].long()
    m = geom.numel() - 1
    last = torch.zeros(s[0].numel(), dtype=torch.bool, device=DEVICE)
    last[ring[1:] - 1] = True
    e = torch.nonzero(~last).flatten()
    row = _rows_of(ring[part[geom]])[e]
    ax, ay, bx, by = s[0][e], s[1][e], s[0][e + 1], s[1][e + 1]
    ex, ey = bx - ax, by - ay
    ll = ex * ex + ey * ey
    out = []
    step = max(1, int(4e7) // e.numel())
    for i in range(0, x.numel(), step):
        px, py = x[i:i + step, None], y[i:i + step, None]
        t = (((px - ax) * ex + (py - ay) * ey) / ll).clamp(0.0, 1.0)
        dist = torch.hypot(ax + t * ex - px, ay + t * ey - py)
        cross = ((ay > py) != (by > py)) & (px < ax + (py - ay) * ex / ey)
        idx = row.expand(px.shape[0], -1)
        best = torch.full((px.shape[0], m), float("inf"), dtype=F64, device=DEVICE).scatter_reduce(1, idx, dist, "amin")
        inside = torch.zeros((px.shape[0], m), dtype=torch.int32, device=DEVICE).scatter_add(1, idx, cross.int()) & 1
        best = torch.where(inside == 1, torch.zeros_like(best), best)
        least = best.amin(1, keepdim=True)
        out.append(best[best == least])
    return torch.cat(out)
