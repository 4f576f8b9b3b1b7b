// Exact polygon x polygon relations beyond intersects: within / contains /
// covers / covered_by / contains_properly / touches / overlaps / crosses for
// two polygonal rows (replaces the DE-9IM mask refine of the reference,
// predicates/polygon.py:19-40, 294-370 and polygon_kernels.py:630-830).
//
// Every boundary edge of one row is cut at the other row's vertices that lie
// on it; between two consecutive cut points the open piece meets the other
// boundary nowhere unless the edges cross properly (reported separately), so
// the location of its midpoint (exact: the midpoint of two fp64 points
// enters every orientation as a sum of two exact determinants) classifies the
// whole piece: interior, exterior, or on the other boundary -- then with the
// other row's interior on the same side or the opposite side (ring
// orientation from the lowest vertex, shells vs holes).  From the pieces of
// both boundaries (A vs B, B vs A):
//   interiors meet     proper crossing, or a piece of one boundary inside the
//                      other, or a shared piece with both interiors on one side
//   A within B (closed) no proper crossing, no piece of dA outside B, no piece
//                      of dB inside A, and every part of A shows a piece inside
//                      B or a same-side shared piece (its interior, which dB
//                      does not enter, is then inside B)
//   A properly in B    A within B and the boundaries never touch
// and within = covered_by, contains = covers (areal rows), touches =
// intersects without interiors meeting, overlaps = interiors meet and neither
// is within the other, crosses = false (two areal rows never cross).
// Valid rings (closed, simple, shells then holes per part) are assumed, as in
// the reference.
#pragma once

#include "vs_distance.h"
#include "vs_exact.h"
#include "vs_internal.h"
#include "vs_polys.h"

namespace vs {

// Exact sign of orient(a, b, p) + orient(a, b, q) = 2 orient(a, b, (p+q)/2),
// orient(a, b, x) = (bx - ax)(xy - ay) - (by - ay)(xx - ax).
__host__ __device__ __noinline__ inline int orient_mid_exact(double ax, double ay, double bx, double by, double px,
                                                             double py, double qx, double qy) {
    double uxh, uxl, uyh, uyl;
    ef_two_diff(bx, ax, uxh, uxl);
    ef_two_diff(by, ay, uyh, uyl);
    ExpAcc acc;
    acc.n = 0;
    const double xs[2] = {px, qx}, ys[2] = {py, qy};
    for (int k = 0; k < 2; ++k) {
        double wxh, wxl, wyh, wyl;
        ef_two_diff(xs[k], ax, wxh, wxl);
        ef_two_diff(ys[k], ay, wyh, wyl);
        acc_add_prod(acc, uxh, wyh);
        acc_add_prod(acc, uxh, wyl);
        acc_add_prod(acc, uxl, wyh);
        acc_add_prod(acc, uxl, wyl);
        acc_add_prod(acc, -uyh, wxh);
        acc_add_prod(acc, -uyh, wxl);
        acc_add_prod(acc, -uyl, wxh);
        acc_add_prod(acc, -uyl, wxl);
    }
    acc.n = ef_compress(acc.e, acc.n);
    return exp_sign(acc.e, acc.n);
}

VS_HD int orient_mid(double ax, double ay, double bx, double by, double px, double py, double qx, double qy) {
    const double ux = bx - ax, uy = by - ay;
    const double t1 = ux * (py - ay), t2 = uy * (px - ax), t3 = ux * (qy - ay), t4 = uy * (qx - ax);
    const double s = (t1 - t2) + (t3 - t4);
    const double bound = 16.0 * kDistEps * (fabs(t1) + fabs(t2) + fabs(t3) + fabs(t4));
    if (s > bound) return 1;
    if (s < -bound) return -1;
    return orient_mid_exact(ax, ay, bx, by, px, py, qx, qy);
}

// Exact sign of (p + q) - 2 c (midpoint coordinate against c).
VS_HD int mid_cmp(double p, double q, double c) {
    double s, t;
    ef_two_sum(p, q, s, t);
    double h, l;
    ef_two_diff(s, 2.0 * c, h, l);
    double e[3];
    int n = 0;
    n = ef_grow(e, n, t);
    n = ef_grow(e, n, l);
    n = ef_grow(e, n, h);
    return exp_sign(e, n);
}

// Location of the midpoint of p and q in polygonal row `row` of P:
// 0 outside, 1 on the boundary, 2 inside (even-odd per part, as the point
// location of the join).
VS_HD int mid_location(double px, double py, double qx, double qy, const Polys& P, int64_t row) {
    // rounded midpoint and a margin beyond its rounding, for cheap skips of
    // edges wholly above, below or left of it (their exact tests agree)
    const double mx = 0.5 * (px + qx), my = 0.5 * (py + qy);
    const double tx = 0x1p-50 * (fabs(px) + fabs(qx)) + 0x1p-1000, ty = 0x1p-50 * (fabs(py) + fabs(qy)) + 0x1p-1000;
    for (int32_t pp = P.geom[row]; pp < P.geom[row + 1]; ++pp) {
        int parity = 0;
        for (int32_t r = P.part[pp]; r < P.part[pp + 1]; ++r)
            for (int32_t c = P.ring[r] + 1; c < P.ring[r + 1]; ++c) {
                const double ax = P.x[c - 1], ay = P.y[c - 1], bx = P.x[c], by = P.y[c];
                if (fmin(ay, by) > my + ty || fmax(ay, by) < my - ty || fmax(ax, bx) < mx - tx) continue;
                const int ya = mid_cmp(py, qy, ay), yb = mid_cmp(py, qy, by);  // sign(2 my - a.y) etc.
                const bool crosses = (ya < 0) != (yb < 0);  // exactly one endpoint above the midpoint
                const bool in_y = (ya >= 0 || yb >= 0) && (ya <= 0 || yb <= 0);
                const bool in_x = (mid_cmp(px, qx, ax) >= 0 || mid_cmp(px, qx, bx) >= 0) &&
                                  (mid_cmp(px, qx, ax) <= 0 || mid_cmp(px, qx, bx) <= 0);
                if (!crosses && !(in_x && in_y)) continue;
                const int o = orient_mid(ax, ay, bx, by, px, py, qx, qy);
                if (o == 0 && in_x && in_y) return 1;
                if (crosses && ((o > 0) == (yb < 0))) parity ^= 1;  // b above: edge goes up
            }
        if (parity) return 2;
    }
    return 0;
}

// Interior of the polygon on the left of ring r's direction: shells counter-
// clockwise, holes clockwise.  The turn at the lowest (then leftmost) vertex
// of a simple ring has the ring's orientation.
VS_HD bool ring_interior_left(const Polys& P, int32_t r, bool shell) {
    const int32_t c0 = P.ring[r], c1 = P.ring[r + 1] - 1;  // last coordinate closes the ring
    const int32_t m = c1 - c0;
    if (m < 3) return shell;
    int32_t k = c0;
    for (int32_t c = c0 + 1; c < c1; ++c)
        if (P.y[c] < P.y[k] || (P.y[c] == P.y[k] && P.x[c] < P.x[k])) k = c;
    int32_t a = k, b = k;  // neighbours distinct from the vertex (repeated points skipped)
    for (int32_t s = 1; s < m; ++s) {
        a = c0 + ((k - c0 - s) % m + m) % m;
        if (P.x[a] != P.x[k] || P.y[a] != P.y[k]) break;
    }
    for (int32_t s = 1; s < m; ++s) {
        b = c0 + (k - c0 + s) % m;
        if (P.x[b] != P.x[k] || P.y[b] != P.y[k]) break;
    }
    const bool ccw = orient2d(P.x[a], P.y[a], P.x[k], P.y[k], P.x[b], P.y[b]) > 0;
    return shell ? ccw : !ccw;
}

struct RelSide {
    bool cross;     // some edges cross properly
    bool touch;     // the boundaries meet (filled by the first pass only)
    bool in_int;    // a boundary piece of X lies in the interior of Y
    bool in_ext;    // a boundary piece of X lies outside Y
    bool same;      // a shared piece with both interiors on one side
    bool all_in;    // every part of X shows a piece inside Y or a same-side shared piece
};

// (nx, ny) = the next vertex of Y strictly between cur and b on edge (a, b)
// (nearest to cur; returns true), or b (returns false).  `ax_major`: compare
// along x (else y).
VS_HD bool next_cut(double ax, double ay, double bx, double by, double cx, double cy, const Polys& Y, int64_t ry,
                    bool ax_major, double& nx, double& ny) {
    nx = bx;
    ny = by;
    bool cut = false;
    const bool inc = ax_major ? bx > ax : by > ay;
    const int32_t v0 = Y.ring[Y.part[Y.geom[ry]]], v1 = Y.ring[Y.part[Y.geom[ry + 1]]];
    for (int32_t v = v0; v < v1; ++v) {
        const double x = Y.x[v], y = Y.y[v];
        const double t = ax_major ? x : y, tc = ax_major ? cx : cy, tn = ax_major ? nx : ny;
        const bool after = inc ? (t > tc && t < tn) : (t < tc && t > tn);
        if (!after) continue;
        if (fmin(ax, bx) > x || x > fmax(ax, bx) || fmin(ay, by) > y || y > fmax(ay, by)) continue;
        if (orient2d(ax, ay, bx, by, x, y) != 0) continue;
        nx = x;
        ny = y;
        cut = true;
    }
    return cut;
}

// One boundary edge c of X (ring interior on the left when left_x) against
// row ry of Y: crossings, contact (when `first`), and its pieces.
VS_HD void relate_edge(const Polys& X, int32_t c, bool left_x, const Polys& Y, int64_t ry, bool first, RelSide& S,
                       bool& part_in) {
    const double ax = X.x[c - 1], ay = X.y[c - 1], bx = X.x[c], by = X.y[c];
    if (ax == bx && ay == by) return;
    // proper crossings (and, on the first pass, any contact)
    for (int32_t q = Y.part[Y.geom[ry]]; q < Y.part[Y.geom[ry + 1]]; ++q)
        for (int32_t d = Y.ring[q] + 1; d < Y.ring[q + 1]; ++d) {
            const double cx = Y.x[d - 1], cy = Y.y[d - 1], dx = Y.x[d], dy = Y.y[d];
            if (fmax(ax, bx) < fmin(cx, dx) || fmax(cx, dx) < fmin(ax, bx) || fmax(ay, by) < fmin(cy, dy) ||
                fmax(cy, dy) < fmin(ay, by))
                continue;
            if (first && !S.touch && segments_touch(ax, ay, bx, by, cx, cy, dx, dy)) S.touch = true;
            const int o1 = orient2d(ax, ay, bx, by, cx, cy), o2 = orient2d(ax, ay, bx, by, dx, dy);
            if (o1 * o2 >= 0) continue;
            const int o3 = orient2d(cx, cy, dx, dy, ax, ay), o4 = orient2d(cx, cy, dx, dy, bx, by);
            if (o3 * o4 < 0) S.cross = true;
        }
    // pieces between consecutive cut points; the last one ends where no cut is
    // left, which also ends the walk along an edge to a NaN (equal to nothing)
    const bool ax_major = ax != bx;
    double px = ax, py = ay;
    for (bool more = true; more;) {
        double qx, qy;
        more = next_cut(ax, ay, bx, by, px, py, Y, ry, ax_major, qx, qy);
        const int loc = mid_location(px, py, qx, qy, Y, ry);
        if (loc == 2) {
            S.in_int = true;
            part_in = true;
        } else if (loc == 0) {
            S.in_ext = true;
        } else {
            // the Y edge holding the midpoint: interiors on one side?
            const double mx = 0.5 * (px + qx), my = 0.5 * (py + qy);
            const double tx = 0x1p-50 * (fabs(px) + fabs(qx)) + 0x1p-1000;
            const double ty = 0x1p-50 * (fabs(py) + fabs(qy)) + 0x1p-1000;
            bool found = false;
            for (int32_t q = Y.part[Y.geom[ry]]; q < Y.part[Y.geom[ry + 1]] && !found; ++q)
                for (int32_t d = Y.ring[q] + 1; d < Y.ring[q + 1]; ++d) {
                    const double cx = Y.x[d - 1], cy = Y.y[d - 1], dx = Y.x[d], dy = Y.y[d];
                    if (cx == dx && cy == dy) continue;
                    if (fmin(cx, dx) > mx + tx || fmax(cx, dx) < mx - tx || fmin(cy, dy) > my + ty ||
                        fmax(cy, dy) < my - ty)
                        continue;
                    if (orient_mid(cx, cy, dx, dy, px, py, qx, qy) != 0) continue;
                    if (mid_cmp(px, qx, fmin(cx, dx)) < 0 || mid_cmp(px, qx, fmax(cx, dx)) > 0 ||
                        mid_cmp(py, qy, fmin(cy, dy)) < 0 || mid_cmp(py, qy, fmax(cy, dy)) > 0)
                        continue;
                    // X's piece lies on this Y edge; ring q's role: the first
                    // ring of its part is the shell
                    found = true;
                    int32_t qp = Y.geom[ry];
                    while (qp + 1 < Y.geom[ry + 1] && Y.part[qp + 1] <= q) ++qp;
                    const bool ly = ring_interior_left(Y, q, q == Y.part[qp]);
                    const bool same_dir = dot_diff_sign(bx, ax, by, ay, dx, cx, dy, cy) > 0;
                    if (same_dir ? (ly == left_x) : (ly != left_x)) {
                        S.same = true;
                        part_in = true;
                    }
                    break;
                }
        }
        px = qx;
        py = qy;
    }
}

// Pieces of X's boundary against row ry of Y.
VS_HD RelSide relate_side(const Polys& X, int64_t rx, const Polys& Y, int64_t ry, bool first) {
    RelSide S = {false, false, false, false, false, true};
    for (int32_t pp = X.geom[rx]; pp < X.geom[rx + 1]; ++pp) {
        bool part_in = false;
        for (int32_t r = X.part[pp]; r < X.part[pp + 1]; ++r) {
            const bool left_x = ring_interior_left(X, r, r == X.part[pp]);
            for (int32_t c = X.ring[r] + 1; c < X.ring[r + 1]; ++c) relate_edge(X, c, left_x, Y, ry, first, S, part_in);
        }
        if (!part_in) S.all_in = false;
    }
    return S;
}

struct Relation {
    bool interiors_meet;
    bool a_in_b;         // A within B (closed)
    bool b_in_a;         // B within A (closed)
    bool touch;          // the boundaries meet
};

// The relation from the pieces of both boundaries (sa: A's pieces, with the
// contact of the boundaries; sb: B's).
VS_HD Relation merge_sides(const RelSide& sa, const RelSide& sb) {
    Relation R;
    const bool cross = sa.cross || sb.cross;
    R.interiors_meet = cross || sa.in_int || sb.in_int || sa.same || sb.same;
    R.a_in_b = !cross && !sa.in_ext && !sb.in_int && sa.all_in;
    R.b_in_a = !cross && !sb.in_ext && !sa.in_int && sb.all_in;
    R.touch = sa.touch;
    return R;
}

VS_HD Relation relate_polygons(const Polys& A, int64_t ra, const Polys& B, int64_t rb) {
    const RelSide sa = relate_side(A, ra, B, rb, true);
    return merge_sides(sa, relate_side(B, rb, A, ra, false));
}

VS_HD double4 row_box(const Polys& P, int64_t row) {
    double4 b = make_double4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (int32_t c = P.ring[P.part[P.geom[row]]]; c < P.ring[P.part[P.geom[row + 1]]]; ++c) {
        b.x = fmin(b.x, P.x[c]);
        b.y = fmin(b.y, P.y[c]);
        b.z = fmax(b.z, P.x[c]);
        b.w = fmax(b.w, P.y[c]);
    }
    return b;
}

// Some edge of A crosses some edge of B properly (interior points of both).
VS_HD bool any_proper_crossing(const Polys& A, int64_t ra, const Polys& B, int64_t rb) {
    for (int32_t r = A.part[A.geom[ra]]; r < A.part[A.geom[ra + 1]]; ++r)
        for (int32_t c = A.ring[r] + 1; c < A.ring[r + 1]; ++c) {
            const double ax = A.x[c - 1], ay = A.y[c - 1], bx = A.x[c], by = A.y[c];
            for (int32_t q = B.part[B.geom[rb]]; q < B.part[B.geom[rb + 1]]; ++q)
                for (int32_t d = B.ring[q] + 1; d < B.ring[q + 1]; ++d) {
                    const double cx = B.x[d - 1], cy = B.y[d - 1], dx = B.x[d], dy = B.y[d];
                    if (fmax(ax, bx) < fmin(cx, dx) || fmax(cx, dx) < fmin(ax, bx) || fmax(ay, by) < fmin(cy, dy) ||
                        fmax(cy, dy) < fmin(ay, by))
                        continue;
                    if (orient2d(ax, ay, bx, by, cx, cy) * orient2d(ax, ay, bx, by, dx, dy) >= 0) continue;
                    if (orient2d(cx, cy, dx, dy, ax, ay) * orient2d(cx, cy, dx, dy, bx, by) < 0) return true;
                }
        }
    return false;
}

// predicate from the full relation (intersects already known for touches).
VS_HD bool relation_decides(int pred, const Relation& R) {
    switch (pred) {
        case VS_PRED_WITHIN:
        case VS_PRED_COVERED_BY: return R.a_in_b;
        case VS_PRED_CONTAINS:
        case VS_PRED_COVERS: return R.b_in_a;
        case VS_PRED_CONTAINS_PROPERLY: return R.b_in_a && !R.touch;
        case VS_PRED_TOUCHES: return !R.interiors_meet;
        case VS_PRED_OVERLAPS: return R.interiors_meet && !R.a_in_b && !R.b_in_a;
        default: return false;
    }
}

// Cheap necessary conditions of predicate(A row, B row) for two polygonal
// rows (codes of vsjoin.h): box containment for the containment predicates;
// intersects, then a proper crossing -- which settles every relation -- for
// touches / overlaps.  1 true, 0 false; undecided (intersects is known to hold
// for touches then): -2 when one row's box lies strictly inside the other's,
// else -1.  A polygon whose boundary does not meet another's lies strictly
// inside it, box and all, or outside, so -1 means that the boundaries touch (or
// that a row has several parts) and only the full relation can decide.
__device__ inline int polygon_predicate_fast(int pred, const Polys& A, int64_t ra, const Polys& B, int64_t rb) {
    if (pred == VS_PRED_INTERSECTS) return polygons_intersect_auto(A, ra, B, rb) ? 1 : 0;
    if (pred == VS_PRED_CROSSES) return 0;
    const bool inclusion = pred != VS_PRED_TOUCHES && pred != VS_PRED_OVERLAPS;
    const bool a_inner = pred == VS_PRED_WITHIN || pred == VS_PRED_COVERED_BY;
    double4 in, out;
    if (inclusion) {
        in = a_inner ? row_box(A, ra) : row_box(B, rb);
        out = a_inner ? row_box(B, rb) : row_box(A, ra);
        if (!(out.x <= in.x && in.z <= out.z && out.y <= in.y && in.w <= out.w)) return 0;
    } else if (!polygons_intersect_auto(A, ra, B, rb)) {
        return 0;
    }
    if (any_proper_crossing(A, ra, B, rb)) return pred == VS_PRED_OVERLAPS ? 1 : 0;
    if (!inclusion) {
        in = row_box(A, ra);
        out = row_box(B, rb);
    }
    const bool nested = (out.x < in.x && in.z < out.z && out.y < in.y && in.w < out.w) ||
                        (in.x < out.x && out.z < in.z && in.y < out.y && out.w < in.w);
    return nested ? -2 : -1;
}

// ---------------------------------------------------------------------------
// One wave per pair, for pairs of large rows.
// ---------------------------------------------------------------------------
// One wave's LDS for wave_edge_pairs.
constexpr int kEdgeTile = 128;
struct WaveEdgeLds {
    int32_t a[kEdgeTile];     // A edges near B (their end coordinate)
    int32_t b[kEdgeTile];     // a tile of B edges near A's current edges
    float4 box[kEdgeTile];    // their boxes (min x, min y, max x, max y)
    int32_t qa[kEdgeTile], qb[kEdgeTile];  // edge pairs whose boxes meet
};

// Boxes in fp32, every bound rounded to nearest.  Rounding is monotone, so
// boxes that meet in fp64 meet in fp32: the tests on them only drop pairs that
// cannot touch, and the exact tests see every other pair.
__device__ __forceinline__ float4 edge_box_f32(const Polys& P, int32_t c) {
    const float ax = (float)P.x[c - 1], ay = (float)P.y[c - 1], bx = (float)P.x[c], by = (float)P.y[c];
    return make_float4(fminf(ax, bx), fminf(ay, by), fmaxf(ax, bx), fmaxf(ay, by));
}

__device__ __forceinline__ bool boxes_meet(const float4& a, const float4& b) {
    return !(a.z < b.x || b.z < a.x || a.w < b.y || b.w < a.y);
}

__device__ __forceinline__ float4 wave_union(float4 b) {
    for (int o = 32; o > 0; o >>= 1) {
        b.x = fminf(b.x, __shfl_xor(b.x, o, 64));
        b.y = fminf(b.y, __shfl_xor(b.y, o, 64));
        b.z = fmaxf(b.z, __shfl_xor(b.z, o, 64));
        b.w = fmaxf(b.w, __shfl_xor(b.w, o, 64));
    }
    return b;
}

__device__ __forceinline__ float4 box_cut(const float4& a, const float4& b) {
    return make_float4(fmaxf(a.x, b.x), fmaxf(a.y, b.y), fminf(a.z, b.z), fminf(a.w, b.w));
}

__device__ __forceinline__ float4 empty_box_f32() { return make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY); }

// Box of the coordinates [s.lo, s.hi), in fp32, by one wave.
__device__ inline float4 wave_row_box_f32(const Polys& P, const RowSpan& s, int lane) {
    float4 b = empty_box_f32();
    for (int32_t c = s.lo + lane; c < s.hi; c += 64) {
        const float x = (float)P.x[c], y = (float)P.y[c];
        b = make_float4(fminf(b.x, x), fminf(b.y, y), fmaxf(b.z, x), fmaxf(b.w, y));
    }
    return wave_union(b);
}

// How two segments meet: 0 not at all, 1 they touch (segments_touch), 2 they
// cross in interior points of both.
VS_HD int segment_contact(double ax, double ay, double bx, double by, double cx, double cy, double dx, double dy) {
    if (fmax(ax, bx) < fmin(cx, dx) || fmax(cx, dx) < fmin(ax, bx) || fmax(ay, by) < fmin(cy, dy) ||
        fmax(cy, dy) < fmin(ay, by))
        return 0;
    const int o1 = orient2d(ax, ay, bx, by, cx, cy);
    const int o2 = orient2d(ax, ay, bx, by, dx, dy);
    const int o3 = orient2d(cx, cy, dx, dy, ax, ay);
    const int o4 = orient2d(cx, cy, dx, dy, bx, by);
    if (o1 * o2 < 0 && o3 * o4 < 0) return 2;
    if (o1 == 0 && cx >= fmin(ax, bx) && cx <= fmax(ax, bx) && cy >= fmin(ay, by) && cy <= fmax(ay, by)) return 1;
    if (o2 == 0 && dx >= fmin(ax, bx) && dx <= fmax(ax, bx) && dy >= fmin(ay, by) && dy <= fmax(ay, by)) return 1;
    if (o3 == 0 && ax >= fmin(cx, dx) && ax <= fmax(cx, dx) && ay >= fmin(cy, dy) && ay <= fmax(cy, dy)) return 1;
    if (o4 == 0 && bx >= fmin(cx, dx) && bx <= fmax(cx, dx) && by >= fmin(cy, dy) && by <= fmax(cy, dy)) return 1;
    return 0;
}

// The closest contact over the edge pairs of two rows, by one wave (every lane
// returns it): 2 some pair crosses, 1 some pair touches and none crosses, 0
// neither; returns at the first contact of at least `enough`.  ba / bb: the
// rows' fp32 boxes.
//
// Only edges that meet both rows' boxes can touch, and of those few meet each
// other, so: A's edges near B's box are listed and taken 64 at a time, one per
// lane (fewer: each edge gets several lanes, which share B's edges); B's edges
// near them are collected in LDS tiles as fp32 boxes; box pairs that meet are
// queued, and a full queue gets the exact test with all lanes at work.  Testing
// every edge pair of the rows in fp64, with a wave waiting for any lane's exact
// test, took 11.1 ms for 600k pairs of 57 x 57 coordinates; this takes 2.0 ms,
// and rows without contact need no full relation (2.9 ms for the 3% that did).
// Bound by latency: 412M vector and 409M scalar instructions (some 690 of each a
// pair) keep the vector units busy a third of the time at 3.2 waves a SIMD; the
// rest waits for the chain of offset loads and the LDS lists' order points.
__device__ inline int wave_edge_pairs(const Polys& A, const RowSpan& sa, const float4& ba, const Polys& B,
                                      const RowSpan& sb, const float4& bb, int enough, WaveEdgeLds& W, int lane) {
    const float4 both = box_cut(ba, bb);
    const uint64_t lt = lanemask_lt();
    int found = 0, nq = 0;
    // exact tests of the first `n` (at most 64) queued pairs
    auto test_queue = [&](int n) {
        wave_lds_order();
        int k = 0;
        if (lane < n) {
            const int32_t c = W.qa[lane], d = W.qb[lane];
            k = segment_contact(A.x[c - 1], A.y[c - 1], A.x[c], A.y[c], B.x[d - 1], B.y[d - 1], B.x[d], B.y[d]);
        }
        if (__ballot(k == 2)) found = 2;
        else if (found < 1 && __ballot(k == 1)) found = 1;
    };
    int na = 0;
    for (int32_t a0 = sa.lo + 1; a0 < sa.hi; a0 += 64) {
        {
            const int32_t c = a0 + lane;
            const bool near = is_row_edge(A, sa, c) && boxes_meet(edge_box_f32(A, c), both);
            const uint64_t m = __ballot(near);
            if (near) W.a[na + __popcll(m & lt)] = c;
            na += __popcll(m);
        }
        const bool last = a0 + 64 >= sa.hi;
        while (na >= 64 || (last && na > 0)) {
            wave_lds_order();
            const int n = na < 64 ? na : 64;
            int width = 1;  // lanes per pass over A's edges; 64 / width share each B tile
            while (width < n) width <<= 1;
            const int ai = lane & (width - 1), sub = lane / width, subs = 64 / width;
            const bool has = ai < n;
            const int32_t ca = W.a[has ? ai : 0];
            const float4 abox = edge_box_f32(A, ca);
            // several passes over A: each one's edges are consecutive along
            // the rings, so B is filtered by their own box
            const float4 lim = na == n && last && a0 == sa.lo + 1 ? both : box_cut(wave_union(abox), bb);
            int nb = 0;
            for (int32_t b0 = sb.lo + 1; b0 < sb.hi; b0 += 64) {
                const int32_t d = b0 + lane;
                float4 dbox = empty_box_f32();
                bool near = is_row_edge(B, sb, d);
                if (near) {
                    dbox = edge_box_f32(B, d);
                    near = boxes_meet(dbox, lim);
                }
                const uint64_t m = __ballot(near);
                if (near) {
                    const int slot = nb + __popcll(m & lt);
                    W.b[slot] = d;
                    W.box[slot] = dbox;
                }
                nb += __popcll(m);
                if (nb <= 64 && b0 + 64 < sb.hi) continue;  // room for another 64
                wave_lds_order();
                for (int k0 = 0; k0 < nb; k0 += subs) {
                    const int k = k0 + sub;
                    const bool hit = has && k < nb && boxes_meet(abox, W.box[k < nb ? k : 0]);
                    const uint64_t h = __ballot(hit);
                    if (!h) continue;
                    if (hit) {
                        const int slot = nq + __popcll(h & lt);
                        W.qa[slot] = ca;
                        W.qb[slot] = W.b[k];
                    }
                    nq += __popcll(h);
                    if (nq >= 64) {
                        test_queue(64);
                        if (found >= enough) return found;
                        nq -= 64;
                        int32_t ma = 0, mb = 0;
                        if (lane < nq) {
                            ma = W.qa[64 + lane];
                            mb = W.qb[64 + lane];
                        }
                        wave_lds_order();
                        if (lane < nq) {
                            W.qa[lane] = ma;
                            W.qb[lane] = mb;
                        }
                        wave_lds_order();
                    }
                }
                wave_lds_order();
                nb = 0;
            }
            na -= n;
            const int32_t rest = lane < na ? W.a[64 + lane] : 0;
            wave_lds_order();
            if (lane < na) W.a[lane] = rest;
            wave_lds_order();
        }
    }
    if (nq > 0) test_queue(nq);
    return found;
}

// The point lies inside the row of P or on its boundary, by one wave.
__device__ inline bool wave_not_outside(double px, double py, const Polys& P, int64_t row, int lane) {
    for (int32_t pp = P.geom[row]; pp < P.geom[row + 1]; ++pp) {
        const RowSpan t = {P.ring[P.part[pp]], P.ring[P.part[pp + 1]], P.part[pp], P.part[pp + 1]};
        int parity = 0;
        bool on = false;
        for (int32_t c0 = t.lo + 1; c0 < t.hi; c0 += 64) {
            const int32_t c = c0 + lane;
            if (is_row_edge(P, t, c)) on |= edge_step_f64(px, py, P.x[c - 1], P.y[c - 1], P.x[c], P.y[c], parity) != 0;
        }
        if (__ballot(on) != 0 || (__popcll(__ballot(parity)) & 1)) return true;
    }
    return false;
}

// Some ring of row ra of A starts at a point of row rb of B (not outside).
__device__ inline bool wave_rings_start_in(const Polys& A, const RowSpan& sa, const Polys& B, int64_t rb,
                                           const float4& bb, int lane) {
    for (int32_t r = sa.r0; r < sa.r1; ++r) {
        const int32_t c = A.ring[r];
        if (A.ring[r + 1] <= c) continue;
        const double x = A.x[c], y = A.y[c];
        const float fx = (float)x, fy = (float)y;
        if (fx < bb.x || fx > bb.z || fy < bb.y || fy > bb.w) continue;  // outside B's box
        if (wave_not_outside(x, y, B, rb, lane)) return true;
    }
    return false;
}

__device__ inline double4 wave_row_box(const Polys& P, int64_t row, int lane) {
    double4 b = make_double4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (int32_t c = P.ring[P.part[P.geom[row]]] + lane; c < P.ring[P.part[P.geom[row + 1]]]; c += 64) {
        b.x = fmin(b.x, P.x[c]);
        b.y = fmin(b.y, P.y[c]);
        b.z = fmax(b.z, P.x[c]);
        b.w = fmax(b.w, P.y[c]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        b.x = fmin(b.x, __shfl_xor(b.x, o, 64));
        b.y = fmin(b.y, __shfl_xor(b.y, o, 64));
        b.z = fmax(b.z, __shfl_xor(b.z, o, 64));
        b.w = fmax(b.w, __shfl_xor(b.w, o, 64));
    }
    return b;
}

// ring_interior_left by one wave (every lane returns the answer): lanes scan
// strided vertices for the lowest (then leftmost, then first) one and a
// shuffle reduction picks it -- the vertex the serial scan finds.
__device__ inline bool wave_ring_interior_left(const Polys& P, int32_t r, bool shell, int lane) {
    const int32_t c0 = P.ring[r], c1 = P.ring[r + 1] - 1;  // last coordinate closes the ring
    const int32_t m = c1 - c0;
    if (m < 3) return shell;
    int32_t k = c1;  // c1: no vertex yet
    double ky = INFINITY, kx = INFINITY;
    for (int32_t c = c0 + lane; c < c1; c += 64) {
        const double y = P.y[c], x = P.x[c];
        if (k == c1 || y < ky || (y == ky && x < kx)) {
            k = c;
            ky = y;
            kx = x;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const int32_t k2 = __shfl_xor(k, o, 64);
        const double y2 = __shfl_xor(ky, o, 64), x2 = __shfl_xor(kx, o, 64);
        if (k2 != c1 && (k == c1 || y2 < ky || (y2 == ky && (x2 < kx || (x2 == kx && k2 < k))))) {
            k = k2;
            ky = y2;
            kx = x2;
        }
    }
    k = __shfl(k, 0, 64);  // one vertex for every lane (NaN coordinates compare unordered)
    int32_t a = k, b = k;  // neighbours distinct from the vertex (repeated points skipped)
    for (int32_t s = 1; s < m; ++s) {
        a = c0 + ((k - c0 - s) % m + m) % m;
        if (P.x[a] != P.x[k] || P.y[a] != P.y[k]) break;
    }
    for (int32_t s = 1; s < m; ++s) {
        b = c0 + (k - c0 + s) % m;
        if (P.x[b] != P.x[k] || P.y[b] != P.y[k]) break;
    }
    const bool ccw = orient2d(P.x[a], P.y[a], P.x[k], P.y[k], P.x[b], P.y[b]) > 0;
    return shell ? ccw : !ccw;
}

// relate_side by one wave: lanes split each ring's edges, votes merge.
__device__ inline RelSide wave_relate_side(const Polys& X, int64_t rx, const Polys& Y, int64_t ry, bool first,
                                           int lane) {
    RelSide S = {false, false, false, false, false, true};
    bool all_in = true;
    for (int32_t pp = X.geom[rx]; pp < X.geom[rx + 1]; ++pp) {
        bool part_in = false;
        for (int32_t r = X.part[pp]; r < X.part[pp + 1]; ++r) {
            const bool left_x = wave_ring_interior_left(X, r, r == X.part[pp], lane);
            for (int32_t c = X.ring[r] + 1 + lane; c < X.ring[r + 1]; c += 64)
                relate_edge(X, c, left_x, Y, ry, first, S, part_in);
        }
        if (__ballot(part_in) == 0) all_in = false;
    }
    RelSide W;
    W.cross = __ballot(S.cross) != 0;
    W.touch = __ballot(S.touch) != 0;
    W.in_int = __ballot(S.in_int) != 0;
    W.in_ext = __ballot(S.in_ext) != 0;
    W.same = __ballot(S.same) != 0;
    W.all_in = all_in;
    return W;
}

__device__ inline Relation wave_relate_polygons(const Polys& A, int64_t ra, const Polys& B, int64_t rb, int lane) {
    const RelSide sa = wave_relate_side(A, ra, B, rb, true, lane);
    return merge_sides(sa, wave_relate_side(B, rb, A, ra, false, lane));
}

// One side of the relation of two rows whose boundaries do not meet: every
// ring of A then lies in one piece inside or outside B, where its first vertex
// does.  A ring without two distinct points has no piece.
__device__ inline RelSide wave_apart_side(const Polys& A, int64_t ra, const Polys& B, int64_t rb, const float4& bb,
                                          int lane) {
    RelSide S = {false, false, false, false, false, true};
    for (int32_t pp = A.geom[ra]; pp < A.geom[ra + 1]; ++pp) {
        bool part_in = false;
        for (int32_t r = A.part[pp]; r < A.part[pp + 1]; ++r) {
            const int32_t c0 = A.ring[r], c1 = A.ring[r + 1];
            if (c1 <= c0) continue;
            const double x = A.x[c0], y = A.y[c0];
            bool piece = false;
            for (int32_t c = c0 + 1; c < c1 && !piece; c += 64)
                piece = __ballot(c + lane < c1 && (A.x[c + lane] != x || A.y[c + lane] != y)) != 0;
            if (!piece) continue;
            const float fx = (float)x, fy = (float)y;
            const bool in =
                !(fx < bb.x || fx > bb.z || fy < bb.y || fy > bb.w) && wave_not_outside(x, y, B, rb, lane);
            S.in_int |= in;
            S.in_ext |= !in;
            part_in |= in;
        }
        S.all_in &= part_in;
    }
    return S;
}

// polygon_predicate_fast by one wave (every lane returns the answer); rows
// whose boundaries do not meet are decided for good.
__device__ inline int wave_polygon_predicate_fast(int pred, const Polys& A, int64_t ra, const Polys& B, int64_t rb,
                                                  WaveEdgeLds& W, int lane) {
    if (pred == VS_PRED_CROSSES) return 0;
    const RowSpan sa = row_span(A, ra), sb = row_span(B, rb);
    const bool inclusion = pred == VS_PRED_WITHIN || pred == VS_PRED_COVERED_BY || pred == VS_PRED_CONTAINS ||
                           pred == VS_PRED_COVERS || pred == VS_PRED_CONTAINS_PROPERLY;
    if (inclusion) {
        const bool a_inner = pred == VS_PRED_WITHIN || pred == VS_PRED_COVERED_BY;
        const double4 in = a_inner ? wave_row_box(A, ra, lane) : wave_row_box(B, rb, lane);
        const double4 out = a_inner ? wave_row_box(B, rb, lane) : wave_row_box(A, ra, lane);
        if (!(out.x <= in.x && in.z <= out.z && out.y <= in.y && in.w <= out.w)) return 0;
    } else if (sa.hi <= sa.lo || sb.hi <= sb.lo) {
        return 0;  // an empty row meets nothing
    }
    const float4 ba = wave_row_box_f32(A, sa, lane), bb = wave_row_box_f32(B, sb, lane);
    // the smaller row's edges go to the lanes
    const int enough = pred == VS_PRED_INTERSECTS ? 1 : 2;
    const int contact = sa.hi - sa.lo <= sb.hi - sb.lo ? wave_edge_pairs(A, sa, ba, B, sb, bb, enough, W, lane)
                                                       : wave_edge_pairs(B, sb, bb, A, sa, ba, enough, W, lane);
    if (contact == 2) return inclusion || pred == VS_PRED_TOUCHES ? 0 : 1;
    if (!inclusion) {
        // without contact the rows meet only if a ring of one starts in the other
        const bool meet = contact == 1 || wave_rings_start_in(A, sa, B, rb, bb, lane) ||
                          wave_rings_start_in(B, sb, A, ra, ba, lane);
        if (!meet || pred == VS_PRED_INTERSECTS) return meet ? 1 : 0;
    }
    if (contact == 1) return -1;
    const RelSide ea = wave_apart_side(A, ra, B, rb, bb, lane), eb = wave_apart_side(B, rb, A, ra, ba, lane);
    return relation_decides(pred, merge_sides(ea, eb)) ? 1 : 0;
}

}  // namespace vs
