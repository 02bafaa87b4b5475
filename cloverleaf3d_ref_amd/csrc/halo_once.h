// The reflective boundary of update_halo_kernel.f90 in one pass.
//
// The reference refreshes a field's y faces, then its x faces, then its z
// faces, each pass reading what the ones before it wrote (bottom/top,
// left/right, back/front; update_halo_kernel.f90:115-1425).  Run as three
// launches, a small mesh spends more time between them than in them.  Here
// every halo cell is written once, by the last pass that covers it, and its
// value is traced back through the passes to the memory the exchange started
// from: a reflection in y of a reflection in x of a reflection in z is one
// interior cell with a sign.
//
// Every cell a trace ends at must keep its old value until it is read.  On a
// tile at least 3 cells thick along every axis the traced-back coordinate is
// interior on every axis whose pass wrote the cell, so the end is no halo cell
// of a refreshed face, with one exception: the last z pass of the x and y face
// fields stops one face short (vol/mass_flux_x: x_max+1+depth, _y:
// y_max+1+depth), and the cells beyond keep the x (or y) pass's reflection
// of a z-halo value that the z pass has not refreshed yet.  The thread that
// refreshes that z-halo cell also writes those, from the old value, before
// it stores the new one.
//
// Compiles for the host as well, where the tests run it cell by cell in any
// order against the three passes.
#pragma once

#include "layout.h"

namespace clover {

// How a field sits on an axis.  For a face normal to axis a, d = 1..depth:
// halo(W) = sgn * f(R) with
//   CELL  low W=1-d R=d     high W=max+d   R=max+1-d   (cell-centred data)
//   STAG  low W=1-d R=1+d   high W=max+1+d R=max+1-d   (vertex data, face data normal to a)
//   FTAN  low W=1-d R=1+d   high W=max+d   R=max-d     (face data tangential to a)
// and tangential ranges min-depth..max+depth (+ext).
enum { K_CELL = 0, K_STAG = 1, K_FTAN = 2 };

// A field's reflective boundary in one word: kind per axis (2 bits each),
// sign flip per axis, and per face L,R,B,T,K,F the +1 on its first and second
// tangential range.
using HaloCode = unsigned;
__host__ __device__ inline int halo_kind(HaloCode h, int axis) { return (h >> (2 * axis)) & 3; }
__host__ __device__ inline bool halo_neg(HaloCode h, int axis) { return (h >> (6 + axis)) & 1; }
__host__ __device__ inline int halo_ext(HaloCode h, int face, int t) { return (h >> (9 + 2 * face + t)) & 1; }

struct Cell3 {
    int j, k, l;
};

__host__ __device__ inline int idx(const Lay &g, const Cell3 &p) { return idx(g, p.j, p.k, p.l); }

// One coordinate of a cell against the faces of its axis: `halo` if it lies in
// the halo of a refreshed face, which copies coordinate r; the sign flip there;
// over: how far it lies beyond max+depth (a pass along another axis reaches
// over 0, or 1 where its tangential range is one longer).
struct Coord {
    bool halo;
    int face, r, over;
};

__host__ __device__ inline Coord coord_of(HaloCode h, int want, int axis, int depth, int mx, int q)
{
    const int kind = halo_kind(h, axis);
    const bool low = q < 1;
    const int d = low ? 1 - q : q - mx - (kind == K_STAG);
    Coord c;
    c.face = 2 * axis + !low;
    c.halo = d >= 1 && d <= depth && ((want >> c.face) & 1);
    c.r = low ? d + (kind != K_CELL) : mx + (kind != K_FTAN) - d;
    c.over = q - mx - depth;
    return c;
}

template <typename S>
__host__ __device__ inline S signed_of(S v, bool neg)
{
    return neg ? (S)(-1.0 * (double)v) : v;  // the reference multiplies by the sign: -0.0 of a zero
}

// which passes write the cell with coordinates x, y, z
__host__ __device__ inline bool x_writes(HaloCode h, const Coord &x, int yover, int zover)
{
    return x.halo && yover <= halo_ext(h, x.face, 0) && zover <= halo_ext(h, x.face, 1);
}
__host__ __device__ inline bool y_writes(HaloCode h, const Coord &y, int xover, int zover)
{
    return y.halo && xover <= halo_ext(h, y.face, 0) && zover <= halo_ext(h, y.face, 1);
}
__host__ __device__ inline bool z_writes(HaloCode h, const Coord &z, int xover, int yover)
{
    return z.halo && xover <= halo_ext(h, z.face, 0) && yover <= halo_ext(h, z.face, 1);
}

// The cells that keep an x or y reflection of the old value of the z-halo
// cell p (written by the z pass; see above): writes them.
template <typename S>
__host__ __device__ inline void write_stale(const Lay &g, int depth, HaloCode h, int want, S *dst, const Cell3 &p, S old)
{
    const Coord z = coord_of(h, want, 2, depth, g.z_max, p.l);
#pragma unroll 1
    for (int t = 0; t < 2; t++) {
        // t 0: an x-face field's column x_max+1+depth, whose x pass copies p's
        // column; t 1: a y-face field's row y_max+1+depth
        if (halo_kind(h, t) != K_STAG || halo_kind(h, 2) != K_FTAN) continue;
        const int xm = g.x_max, ym = g.y_max, mx = t ? ym : xm, omx = t ? xm : ym;
        const int j = p.j, k = p.k, at = t ? k : j, other = t ? j : k;
        if (at != mx + 1 - depth) continue;
        // itself and its images across the other axis's faces
#pragma unroll 1
        for (int m = 0; m < 3; m++) {
            const int image = m == 0 ? other : m == 1 ? 2 - other : 2 * omx - other;
            if (m && image == other) continue;
            const Cell3 w{t ? image : mx + 1 + depth, t ? mx + 1 + depth : image, p.l};
            const Coord x = coord_of(h, want, 0, depth, g.x_max, w.j), y = coord_of(h, want, 1, depth, g.y_max, w.k);
            if (z_writes(h, z, x.over, y.over)) continue;
            const bool xw = x_writes(h, x, y.over, z.over);
            const bool yw = y_writes(h, y, xw ? 0 : x.over, z.over);
            if (!(xw || yw) || (xw ? x.r : w.j) != p.j || (yw ? y.r : w.k) != p.k) continue;
            dst[idx(g, w)] = signed_of(old, (xw && halo_neg(h, 0)) != (yw && halo_neg(h, 1)));
        }
    }
}

// The move that refreshes a halo cell: from offset src to offset dst, with a
// sign; stale: the cell's old value also goes where write_stale puts it.
struct Move {
    int src, dst;
    bool neg, stale;
};

// The halo cell of the face along `axis` whose coordinates are x, y, z (cell
// p): its move; false if a later pass covers it or it lies outside the field's
// ranges.
__host__ __device__ inline bool halo_move(const Lay &g, int depth, HaloCode h, int axis, const Cell3 &p, const Coord &x,
                                          const Coord &y, const Coord &z, Move &m)
{
    const bool zw = z_writes(h, z, x.over, y.over), xw = x_writes(h, x, y.over, z.over),
               yw = y_writes(h, y, x.over, z.over);
    int j = p.j, k = p.k, l = p.l;
    bool neg = halo_neg(h, axis), mine;
    if (axis == 2) {
        mine = zw;
        l = z.r;  // interior from here on: only the other axis can still be out of a pass's range
        const bool xs = x_writes(h, x, y.over, 0), ys = y_writes(h, y, xs ? 0 : x.over, 0);
        j = xs ? x.r : j;
        k = ys ? y.r : k;
        neg ^= (xs && halo_neg(h, 0)) != (ys && halo_neg(h, 1));
    } else if (axis == 0) {
        j = x.r;
        const bool ys = y_writes(h, y, 0, z.over);
        k = ys ? y.r : k;
        mine = xw && !zw && !z_writes(h, z, 0, ys ? 0 : y.over);  // (the last: write_stale's)
        neg ^= ys && halo_neg(h, 1);
    } else {
        k = y.r;
        mine = yw && !xw && !zw && !z_writes(h, z, x.over, 0);
    }
    m.src = idx(g, j, k, l);
    m.dst = idx(g, p);
    m.neg = neg;
    m.stale = mine && axis == 2 && (p.j == g.x_max + 1 - depth || p.k == g.y_max + 1 - depth);
    return mine;
}

// One thread's share of the face along `axis` (side 0 low, 1 high): its
// `depth` halo cells at tangential coordinates (a, b).
template <typename S>
__host__ __device__ inline void reflect_once(const Lay &g, int depth, HaloCode h, int want, S *dst, int axis, int side, int a,
                                             int b)
{
    const int xm = g.x_max, ym = g.y_max, zm = g.z_max, mx = axis == 0 ? xm : axis == 1 ? ym : zm;
    const int at1 = !side ? 0 : mx + 1 + (halo_kind(h, axis) == K_STAG);
    const Coord ta = coord_of(h, want, axis == 0 ? 1 : 0, depth, axis == 0 ? ym : xm, a),
                tb = coord_of(h, want, axis == 2 ? 1 : 2, depth, axis == 2 ? ym : zm, b);
    Cell3 p[2];
    Move m[2];
    bool mine[2] = {false, false};
    S v[2], old[2];
#pragma unroll
    for (int d = 0; d < 2; d++) {
        if (d >= depth) break;
        const int at = !side ? at1 - d : at1 + d;
        p[d] = Cell3{axis == 0 ? at : a, axis == 0 ? a : axis == 1 ? at : b, axis == 2 ? at : b};
        const Coord c = coord_of(h, want, axis, depth, mx, at);
        mine[d] = axis == 0   ? halo_move(g, depth, h, 0, p[d], c, ta, tb, m[d])
                  : axis == 1 ? halo_move(g, depth, h, 1, p[d], ta, c, tb, m[d])
                              : halo_move(g, depth, h, 2, p[d], ta, tb, c, m[d]);
        // every load before the first store, so that they are in flight together
        if (mine[d]) v[d] = dst[m[d].src];
        if (mine[d] && m[d].stale) old[d] = dst[m[d].dst];
    }
    if ((mine[0] && m[0].stale) || (mine[1] && m[1].stale)) {
#pragma unroll 1
        for (int d = 0; d < 2; d++)
            if (d ? mine[1] && m[1].stale : mine[0] && m[0].stale)
                write_stale(g, depth, h, want, dst, d ? Cell3{p[1].j, p[1].k, p[1].l} : Cell3{p[0].j, p[0].k, p[0].l},
                            d ? S(old[1]) : S(old[0]));
    }
#pragma unroll
    for (int d = 0; d < 2; d++)
        if (mine[d]) dst[m[d].dst] = signed_of(v[d], m[d].neg);
}

}  // namespace clover
