// gdt_hull.h -- a point's ring as a convex hull (host/device): the LDS tile
// kernels' first pass over every point.
//
// Inversion about v, c -> c / |c|^2, maps circles through v to lines, so the
// ring of v is the convex hull of the inverted candidates, in order, and
// "c lies inside circle (v, a, b)" is "c' lies beyond the line a'b'".  The
// hull of a star-shaped polygon (candidates sorted by angle about v) takes a
// few linear passes, where gift wrapping scans the candidates once per
// neighbour, and each lane of a wavefront does about the same amount of work:
//   1. the entries of the 5x5 cell block around v, one 32-bit key each
//      (angle, entry), sorted by a network in registers;
//   2. a pass over the sorted keys that drops every entry b between its kept
//      predecessor a and its successor c with c inside circle (v, a, b) (more than half of
//      them), then Graham's scan over the rest; the nearest entry, which is on
//      the hull, starts the list and stays;
//   3. each ring triangle whose circle leaves the scanned cells scans the
//      circle's other cells (as a step of gdt_tile.h does), and a point found
//      in it is put in: the nearest one along the bisector is the
//      successor of a, itself a neighbour by induction from the start.
// The decision is the sign of the in-circle determinant of the displacements,
//   P = |c|^2 (a x b) - |b|^2 (a x c) + |a|^2 (b x c),
// each new entry costing two cross products.  A point whose block holds too
// many or too few entries, whose entries are not in strict angular order with
// gaps below half a turn (nearly collinear with v beyond the keys'
// resolution), with an exact tie, or with a circle leaving the window is left
// to the steps (HULL_STEPS; nothing of its row is written).
#pragma once

#include "gdt_tile.h"

#include <utility>

#if defined(__HIPCC__)
#define GDT_UNROLL _Pragma("unroll")
#else
#define GDT_UNROLL
#endif

#define GDT_HULL_SLOTS 30     // entries of the block, v included
#define GDT_HULL_WORDS 11     // LDS words per lane: 22 list entries (odd: no bank conflicts;
                              // one more word after the last lane's)
#define GDT_HULL_LIST 22
#define GDT_HULL_RING 12      // longest ring that leaves room for a row table behind it
#define GDT_HULL_TBL 6        // the row table's five words (and the one read after them)
#define GDT_HULL_ROUNDS 64    // triangles of part 3 before a point is left

// List entries (the lane's words also hold a row table).
typedef uint16_t __attribute__((may_alias)) gdt_u16a;

// Any lane of the wave (host builds: the one lane).
GDT_HD inline bool gdt_hull_any(bool b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __any(b);
#else
    return b;
#endif
}

// Sorting network (Batcher's merge exchange, Knuth 5.2.2 algorithm M).
struct GdtNet {
    int n;
    unsigned char a[256], b[256];
};
constexpr GdtNet gdt_make_net(int n)
{
    GdtNet t{};
    int top = 1;
    while (2 * top < n) top *= 2;
    for (int p = top; p > 0; p /= 2) {
        int q = top, r = 0, d = p;
        for (;;) {
            for (int i = 0; i < n - d; ++i)
                if ((i & p) == r) {
                    t.a[t.n] = (unsigned char)i;
                    t.b[t.n] = (unsigned char)(i + d);
                    ++t.n;
                }
            if (q == p) break;
            d = q - p;
            q /= 2;
            r = p;
        }
    }
    return t;
}
constexpr GdtNet GDT_HULL_NET = gdt_make_net(GDT_HULL_SLOTS);

template <size_t I>
GDT_HD inline void gdt_net_step(uint32_t (&k)[GDT_HULL_SLOTS])
{
    constexpr int a = GDT_HULL_NET.a[I], b = GDT_HULL_NET.b[I];
    const uint32_t x = k[a], y = k[b];
    k[a] = x < y ? x : y;
    k[b] = x < y ? y : x;
}
template <size_t... I>
GDT_HD inline void gdt_net_sort(uint32_t (&k)[GDT_HULL_SLOTS], std::index_sequence<I...>)
{
    (gdt_net_step<I>(k), ...);
}

// One entry of the list: displacement and squared length.
struct GdtHullPt {
    double x, y, w;
};

GDT_HD inline double gdt_hull_cross(const GdtHullPt& a, const GdtHullPt& b)
{
    return fma(a.x, b.y, -(a.y * b.x));
}
// P(c) of the circle (v, a, b), from the three cross products.
GDT_HD inline double gdt_hull_p(const GdtHullPt& a, const GdtHullPt& b, const GdtHullPt& c,
                                double ab, double ac, double bc)
{
    return fma(c.w, ab, fma(a.w, bc, -(b.w * ac)));
}

GDT_HD inline int gdt_hull_entry(const uint32_t* words, int i)
{
    return reinterpret_cast<const gdt_u16a*>(words)[i];
}

// The circles against the scanned cells, the rectangle [-hx,hx] x [-hy,hy] of
// cells, as distances from v to its sides.  Circle (v, a, b) has the centre
// q = -K/(2 K0) and R = |q|; with a side's unit normal e at distance D it stays
// inside when R <= D - e.q, that is (e x K)^2 <= 4 K0 D (K0 D + e.K).  (ox, oy):
// v's offset in its cell (GEN: its cell coordinates there).
template <bool GEN>
struct GdtHullBox {
    double nxx, nxy, nyx, nyy;          // unit normals of the cells' sides
    double xm, xp, ym, yp;
    GDT_HD bool holds(const GdtHullPt& a, const GdtHullPt& b) const
    {
        const double k0 = gdt_hull_cross(a, b);
        const double kx = fma(b.w, a.y, -(a.w * b.y)), ky = fma(a.w, b.x, -(b.w * a.x));
        const double ex = GEN ? fma(nxx, kx, nxy * ky) : kx, fx = GEN ? fma(nxx, ky, -(nxy * kx)) : ky;
        const double ey = GEN ? fma(nyx, kx, nyy * ky) : ky, fy = GEN ? fma(nyx, ky, -(nyy * kx)) : kx;
        const double qx = fx * fx * (0.25 * (1. + 1e-6)), qy = fy * fy * (0.25 * (1. + 1e-6));
        auto side = [&](double D, double e, double q) {
            const double kd = k0 * D;
            return q <= kd * (kd + e);
        };
        return side(xp, ex, qx) & side(xm, -ex, qx) & side(yp, ey, qy) & side(ym, -ey, qy) &
               (k0 > 1e-6 * (fabs(a.x * b.y) + fabs(a.y * b.x)));
    }
};
template <bool GEN>
GDT_HD inline GdtHullBox<GEN> gdt_hull_box(const GdtSet& S, double ox, double oy, int hx, int hy)
{
    GdtHullBox<GEN> b;
    b.nxx = GEN ? S.rxx / S.nrx : 1.;
    b.nxy = GEN ? S.rxy / S.nrx : 0.;
    b.nyx = GEN ? S.ryx / S.nry : 0.;
    b.nyy = GEN ? S.ryy / S.nry : 1.;
    const double fx = GEN ? ox * S.bsx : ox, fy = GEN ? oy * S.bsy : oy;   // from the cell's walls
    const double eps = 1e-3 * GDT_FMIN(S.bsx, S.bsy);
    b.xm = fma((double)hx, S.bsx, fx) - eps;
    b.xp = fma((double)(hx + 1), S.bsx, -fx) - eps;
    b.ym = fma((double)hy, S.bsy, fy) - eps;
    b.yp = fma((double)(hy + 1), S.bsy, -fy) - eps;
    return b;
}
// Cells (relative to v's) that circle (v, a, b) can touch, k0 = a x b.
template <bool GEN>
GDT_HD inline void gdt_hull_cells(const GdtSet& S, const GdtHullPt& a, const GdtHullPt& b, double k0,
                                  double ox, double oy, int& x0, int& x1, int& y0, int& y1)
{
    const double kx = fma(b.w, a.y, -(a.w * b.y)), ky = fma(a.w, b.x, -(b.w * a.x));
    const double i2k = gdt_rcp64(2. * k0);
    const double qx = -kx * i2k, qy = -ky * i2k;
    const double rad = gdt_sqrt64(qx * qx + qy * qy) * (1.0 + 1e-9);
    const double mg = 1e-6 * (fabs(qx) + fabs(qy) + rad) + 1e-9 * S.bsx;
    if constexpr (GEN) {
        const double u = ox + fma(S.rxx, qx, S.rxy * qy), ru = (rad + 2. * mg) * S.nrx + 1e-3;
        const double v = oy + fma(S.ryx, qx, S.ryy * qy), rv = (rad + 2. * mg) * S.nry + 1e-3;
        x0 = gdt_cell_floor(u - ru);
        x1 = gdt_cell_floor(u + ru);
        y0 = gdt_cell_floor(v - rv);
        y1 = gdt_cell_floor(v + rv);
    } else {
        gdt_circle_cells<double>(qx - mg, qx + mg, qy - mg, qy + mg, rad, ox, oy, S.ibsx, S.ibsy,
                                 1e-3, x0, x1, y0, y1);
    }
}

// A lane's point while its ring is built: the list's length (entries in the
// lane's LDS words, the nearest first), the ring triangles (i, i + 1) that are not
// certified as a bit mask, whether the point is left to the steps, and the
// level of the scanned block (gdt_hull_build).
struct GdtHull {
    int n, lv;
    uint32_t open;
    bool bad;
    double w0;      // squared distance of the first entry
};

// Parts 1 and 2, and the circles against the scanned cells.  words: the lane's
// GDT_HULL_WORDS LDS words.
template <bool GEN>
GDT_HD inline void gdt_hull_build(const GdtSet& S, const GdtTileLds& L,
                                  const GdtTileLane<double>& st, uint32_t* words, GdtHull& h,
                                  unsigned& npred)
{
    gdt_u16a* lst = reinterpret_cast<gdt_u16a*>(words);
    uint32_t* tbl = words + GDT_HULL_TBL;
    const double vx = st.vx, vy = st.vy;
    auto pt = [&](int k) {
        const gdt_d2 X = L.X64[k];
        GdtHullPt p;
        p.x = X.x - vx;
        p.y = X.y - vy;
        p.w = gdt_dist2_64(p.x, p.y);
        return p;
    };
    // 1. the block's rows, with fewer cells where they hold too many entries:
    // the 5x5 cells (level 0), those without the corners (1), 5x3 (2), 3x3 (3)
    const int r0 = st.c0 - 2 * GDT_WIN;
    auto row_n = [&](int r, int t) {
        return (int)(L.cs[r0 + r * GDT_WIN + 3 - t] - L.cs[r0 + r * GDT_WIN - 2 + t]);
    };
    const int mid = row_n(1, 0) + row_n(2, 0) + row_n(3, 0);
    // (a key holds an entry's distance from the block's first in eight bits)
    const bool wide = L.cs[r0 + 4 * GDT_WIN + 2] - L.cs[r0 - 1] > 255u;
    int lv = 0, ntot = row_n(0, 0) + mid + row_n(4, 0);
    if (ntot > GDT_HULL_SLOTS || wide) {
        lv = 1;
        ntot = row_n(0, 1) + mid + row_n(4, 1);
        if (ntot > GDT_HULL_SLOTS || wide) {
            lv = mid > GDT_HULL_SLOTS ? 3 : 2;
            ntot = lv == 2 ? mid : row_n(1, 1) + row_n(2, 1) + row_n(3, 1);
        }
    }
    const int rb = lv < 2 ? 0 : 1, re = 4 - rb;         // first and last row
    const int te = lv == 1 || lv == 3 ? 1 : 0;          // columns cut from these
    const int tm = lv == 3 ? 1 : 0;                     // and from the rows between
    const uint32_t base = L.cs[r0 + rb * GDT_WIN - 2 + te];
    const uint32_t last = L.cs[r0 + re * GDT_WIN + 3 - te];
    bool ok = ntot <= GDT_HULL_SLOTS && ntot >= 4 && last - base <= 255u;
    int ns = 0;
    for (int r = 0; r < 5; ++r) {
        const int t = r == rb || r == re ? te : tm;
        const uint32_t k = L.cs[r0 + r * GDT_WIN - 2 + t], e = L.cs[r0 + r * GDT_WIN + 3 - t];
        if (r >= rb && r <= re && e > k) tbl[ns++] = k | (e << 16);
    }
    if (!ok) ntot = 0;
    uint32_t key[GDT_HULL_SLOTS];
    float nd2 = 3.0e38f;
    uint32_t nkey = 0;
    {
        const uint32_t* p = tbl;
        uint32_t ke = p[0], wn = p[1];
GDT_UNROLL
        for (int i = 0; i < GDT_HULL_SLOTS; ++i) {
            key[i] = 0xffffffffu;
            if (gdt_hull_any(i < ntot)) {
                if (i < ntot) {
                    const uint32_t k = ke & 0xffffu;
                    const gdt_d2 X = L.X64[k];
                    ++ke;
                    const bool sw = (i + 1 < ntot) & ((ke & 0xffffu) == (ke >> 16));
                    ke = sw ? wn : ke;
                    p += sw ? 1 : 0;
                    wn = p[1];
                    const float x = (float)(X.x - vx), y = (float)(X.y - vy);
                    const float d2 = fmaf(x, x, y * y);
                    // angle in quarter turns from the negative y axis, monotone
                    const float t = y * gdt_rcp32(fabsf(x) + fabsf(y));
                    const float u = GDT_FMAXF(x >= 0.f ? 1.f + t : 3.f - t, 0.f);
                    const uint32_t rel = k - base;
                    if ((int)k != st.iv) {
                        key[i] = ((uint32_t)(u * 4194303.f) << 8) | rel;
                        ok &= d2 > 0.f;      // (a point on v: left to the steps)
                        nkey = d2 < nd2 ? key[i] : nkey;
                        nd2 = GDT_FMINF(nd2, d2);
                    }
                }
            }
        }
    }
    // (squared distances out of FP32's normal range tell no nearest entry: where
    // none was finite the walk began at another one, and 20 to 45 of 1,600 rows
    // were wrong in cells of 1e20 and more)
    ok &= (nd2 > 1.0e-36f) & (nd2 < 3.0e38f);
    // angles counted from the nearest entry's, which comes first as 0 (an entry
    // a key's resolution before it wraps round to the end)
    const uint32_t turn = nkey & ~255u;
GDT_UNROLL
    for (int i = 0; i < GDT_HULL_SLOTS; ++i) {
        const bool used = key[i] != 0xffffffffu;
        const uint32_t k = key[i] == nkey ? 0u : key[i] - turn;
        key[i] = used ? k : 0xffffffffu;
    }
    gdt_net_sort(key, std::make_index_sequence<(size_t)GDT_HULL_NET.n>{});
    // 2. a first pass with the sorted keys in registers: an entry b between its
    // kept predecessor a and its successor c is dropped when c lies inside
    // circle (v, a, b).  bad: an exact tie, or entries not in strict angular
    // order with gaps below half a turn.
    const int n0 = ok ? ntot - 1 : 0;
    bool bad = !ok;
    auto entry = [&](uint32_t k) { return (int)(base + (k & 255u)); };
    const int ks = ok ? entry(nkey) : 0;
    GdtHullPt s0 = pt(ks);
    int n = 1;
    lst[0] = (gdt_u16a)ks;
    {
        GdtHullPt a = s0;
        int kb = ok ? entry(key[1]) : 0;
        GdtHullPt b = pt(kb);
        double ab = gdt_hull_cross(a, b);
        const bool behind = (n0 > 2) & (ab < 0.) & (a.x * b.x + a.y * b.y > 0.);
        if (gdt_hull_any(behind)) {
            // nearly collinear with v and the first entry, but sorted after it
            // by the keys: it comes last
            const uint32_t k1 = key[1];
GDT_UNROLL
            for (int i = 1; i + 1 < GDT_HULL_SLOTS; ++i) {
                const uint32_t next = i + 1 < n0 ? key[i + 1] : (i + 1 == n0 ? k1 : key[i]);
                key[i] = behind ? next : key[i];
            }
            kb = ok ? entry(key[1]) : 0;
            b = pt(kb);
            ab = gdt_hull_cross(a, b);
        }
GDT_UNROLL
        for (int i = 2; i < GDT_HULL_SLOTS; ++i) {
            // (entry i - 1 between a and entry i, or the start after the last)
            if (gdt_hull_any(i <= n0 && !bad)) {
                if (i <= n0) {
                    int kc = i < n0 ? entry(key[i]) : ks;
                    GdtHullPt c = pt(kc);
                    double bc = gdt_hull_cross(b, c), ac = gdt_hull_cross(a, c);
                    if (bc < 0. && i < n0) {
                        // nearly collinear with v and sorted the other way
                        // round by the keys: c comes first
                        const GdtHullPt pb = b;
                        const int ib = kb;
                        const double xb = ab;
                        b = c;
                        c = pb;
                        kb = kc;
                        kc = ib;
                        ab = ac;
                        ac = xb;
                        bc = -bc;
                    }
                    const double P = gdt_hull_p(a, b, c, ab, ac, bc);
                    const bool keep = P > 0.;
                    bad |= !((bc > 0.) & (ab > 0.)) | (P == 0.) | (n >= GDT_HULL_LIST);
                    lst[n < GDT_HULL_LIST ? n : GDT_HULL_LIST - 1] = (gdt_u16a)kb;
                    n += keep ? 1 : 0;
                    a.x = keep ? b.x : a.x;
                    a.y = keep ? b.y : a.y;
                    a.w = keep ? b.w : a.w;
                    ab = keep ? bc : ac;
                    b = c;
                    kb = kc;
                }
            }
        }
    }
    npred += (unsigned)n0;
    bad |= n < 3;
    if (bad) n = 0;
    // then Graham's scan over what is left (the stack grows over the list):
    // a, b its top two entries, c the next entry (the start after the last)
    if (gdt_hull_any(n > 0)) {
        int t = 1, i = 2;       // top of the stack, next entry
        GdtHullPt a = s0, b = pt(lst[1]), c = pt(lst[n > 2 ? 2 : 0]);
        int kc = lst[n > 2 ? 2 : 0];
        double ab = gdt_hull_cross(a, b);
        bool go = n > 0;
        unsigned tests = 0;
        while (gdt_hull_any(go)) {
            if (go) {
                const double bc = gdt_hull_cross(b, c), ac = gdt_hull_cross(a, c);
                const double P = gdt_hull_p(a, b, c, ab, ac, bc);
                const bool push = P > 0. || t == 0;
                bad |= (P == 0.) & (t > 0);
                ++tests;
                // the entry below a, or the one after c
                const int q = push ? (i + 1 < n ? i + 1 : 0) : (t >= 2 ? t - 2 : 0);
                const int kq = lst[q];
                const GdtHullPt x = pt(kq);
                if (push && i < n) lst[t + 1] = (gdt_u16a)kc;
                go = !(push && i >= n) && !bad;
                if (go) {
                    const GdtHullPt oa = a;
                    a.x = push ? b.x : x.x;
                    a.y = push ? b.y : x.y;
                    a.w = push ? b.w : x.w;
                    b.x = push ? c.x : oa.x;
                    b.y = push ? c.y : oa.y;
                    b.w = push ? c.w : oa.w;
                    c.x = push ? x.x : c.x;
                    c.y = push ? x.y : c.y;
                    c.w = push ? x.w : c.w;
                    kc = push ? kq : kc;
                    t += push ? 1 : -1;
                    i += push ? 1 : 0;
                    ab = gdt_hull_cross(a, b);
                }
            }
        }
        npred += tests;
        n = t + 1;
    }
    // 3. the circles against the scanned cells
    double ox, oy;
    if constexpr (GEN) {
        ox = fma(S.rxx, vx, S.rxy * vy) - (double)(st.c0 % GDT_WIN - GDT_FRAME);
        oy = fma(S.ryx, vx, S.ryy * vy) - (double)(st.c0 / GDT_WIN - GDT_FRAME);
    } else {
        ox = gdt_cell_offset(vx, st.c0 % GDT_WIN, S.bsx);
        oy = gdt_cell_offset(vy, st.c0 / GDT_WIN, S.bsy);
    }
    // level 0 and 2: one rectangle; level 1: 5x3 or 3x5; level 3: 3x3
    const GdtHullBox<GEN> box = gdt_hull_box<GEN>(S, ox, oy, lv == 3 ? 1 : 2, lv != 0 ? 1 : 2);
    const GdtHullBox<GEN> box2 = gdt_hull_box<GEN>(S, ox, oy, 1, 2);
    uint32_t open = 0;      // bit i: the triangle (i, i + 1) is not certified
    if (gdt_hull_any(!bad)) {
        double wmin = s0.w;
        bool tie = false;
        int nn = 0;
        if (!bad) {
            GdtHullPt a = s0;
            // (the first vertex is convex, too: the others are already)
            const GdtHullPt z = pt(lst[n - 1]), f = pt(lst[1]);
            const double za = gdt_hull_cross(z, a), zf = gdt_hull_cross(z, f), af = gdt_hull_cross(a, f);
            bad |= !(za > 0.) | !(gdt_hull_p(z, a, f, za, zf, af) > 0.);
            for (int i = 0; i < n; ++i) {
                const GdtHullPt b = i + 1 < n ? pt(lst[i + 1]) : s0;
                bool in = box.holds(a, b);
                if (gdt_hull_any(lv == 1)) in |= (lv == 1) & box2.holds(a, b);
                open |= in ? 0u : 1u << i;
                if (i > 0) {
                    tie |= a.w == wmin;
                    nn = a.w < wmin ? i : nn;
                    wmin = GDT_FMIN(wmin, a.w);
                }
                a = b;
            }
            bad |= tie;
        }
        if (gdt_hull_any(nn != 0 && !bad)) {
            // two nearest entries closer than FP32 told apart: start at the
            // exact one
            if (nn != 0 && !bad) {
                auto reverse = [&](int x, int y) {
                    for (; x < y; ++x, --y) {
                        const gdt_u16a t = lst[x];
                        lst[x] = lst[y];
                        lst[y] = t;
                    }
                };
                reverse(0, nn - 1);
                reverse(nn, n - 1);
                reverse(0, n - 1);
                open = ((open >> nn) | (open << (n - nn))) & ((1u << n) - 1u);
                s0 = pt(lst[0]);
            }
        }
    }
    h.n = n;
    h.lv = lv;
    h.bad = bad | (open != 0 && n > GDT_HULL_RING);
    h.open = h.bad ? 0u : open;
    h.w0 = s0.w;
}

// Part 3 for one triangle (v, a, b) (entries iv, ka, kb; v in window cell c0):
// the circle's cells left of v->a outside the scanned square, cut to part sub
// of W lanes, searched for the point inside it that comes first along the
// bisector.  Returns its entry, -1 if none, -2 if the circle leaves the window
// or an exact tie was met (W > 1: a circle leaving the window is for one
// lane alone).  tbl: the lane's table words.
enum { HULL_NONE = -1, HULL_FAIL = -2 };
template <bool GEN>
GDT_HD inline int gdt_hull_probe(const GdtSet& S, const GdtTileLds& L, int iv, int c0, int lv,
                                 int ka, int kb, uint32_t* tbl, int sub, int W, unsigned& npred)
{
    const gdt_d2 V = L.X64[iv];
    auto pt = [&](int k) {
        const gdt_d2 X = L.X64[k];
        GdtHullPt p;
        p.x = X.x - V.x;
        p.y = X.y - V.y;
        p.w = gdt_dist2_64(p.x, p.y);
        return p;
    };
    const GdtHullPt a = pt(ka);
    GdtHullPt b = pt(kb);
    double k0 = gdt_hull_cross(a, b), ox, oy;
    GdtClip cl;
    if constexpr (GEN) {
        ox = fma(S.rxx, V.x, S.rxy * V.y) - (double)(c0 % GDT_WIN - GDT_FRAME);
        oy = fma(S.ryx, V.x, S.ryy * V.y) - (double)(c0 / GDT_WIN - GDT_FRAME);
        const double au = fma(S.rxx, a.x, S.rxy * a.y), av = fma(S.ryx, a.x, S.ryy * a.y);
        cl = gdt_left_clip(true, (float)au, (float)av, (float)ox, (float)oy, 1.f, 1.f, 1e-3f);
    } else {
        ox = gdt_cell_offset(V.x, c0 % GDT_WIN, S.bsx);
        oy = gdt_cell_offset(V.y, c0 / GDT_WIN, S.bsy);
        cl = gdt_left_clip(true, (float)a.x, (float)a.y, (float)ox, (float)oy, (float)S.bsx,
                           (float)S.bsy, 1e-3f);
    }
    int best = HULL_NONE, hs = lv ? 1 : 2;
    bool tie = false, done = false;
    auto load = [&](int k) { return L.X64[k]; };
    auto visit = [&](int k, const gdt_d2 X) {
        GdtHullPt c;
        c.x = X.x - V.x;
        c.y = X.y - V.y;
        c.w = gdt_dist2_64(c.x, c.y);
        const double ac = gdt_hull_cross(a, c), bc = gdt_hull_cross(b, c);
        const double P = gdt_hull_p(a, b, c, k0, ac, bc);
        if ((ac > 0.) & (P <= 0.) & (k != ka) & (k != kb)) {
            tie |= P == 0.;
            best = k;
            b = c;
            k0 = ac;
        }
    };
    // a circle leaving the window: the 7x7 cells first (they lie in it), then
    // the circle of what they held
    for (int step = 0; step < 2 && !done; ++step) {
        int dx0 = -GDT_SCAN, dx1 = GDT_SCAN, dy0 = -GDT_SCAN, dy1 = GDT_SCAN;
        if (k0 > 1e-6 * (fabs(a.x * b.y) + fabs(a.y * b.x))) {
            int x0, x1, y0, y1;
            gdt_hull_cells<GEN>(S, a, b, k0, ox, oy, x0, x1, y0, y1);
            done = gdt_in_window(S, c0, x0, x1, y0, y1);
            if (done) {
                dx0 = x0;
                dx1 = x1;
                dy0 = y0;
                dy1 = y1;
            }
        }
        if (!done && (step > 0 || W > 1)) break;
        for (int dy = dy0; dy <= dy1;) {
            const unsigned ne = gdt_box_rows(L, c0, dy, dy1, dx0, dx1, hs, cl, tbl, sub, W);
            gdt_scan_tbl(tbl, ne, load, visit);
            npred += ne;
        }
        hs = done ? hs : GDT_SCAN;
    }
    return !done || tie ? HULL_FAIL : best;
}

// Point `k`, found in the circle of triangle i, put into the list; entries
// beside it that are no longer convex go.  Its two triangles are open, but for
// the first where its other vertex stays (the search covered that circle).
GDT_HD inline void gdt_hull_insert(const GdtTileLds& L, int iv, uint32_t* words, GdtHull& h, int i,
                                   int k)
{
    gdt_u16a* lst = reinterpret_cast<gdt_u16a*>(words);
    const gdt_d2 V = L.X64[iv];
    auto pt = [&](int e) {
        const gdt_d2 X = L.X64[e];
        GdtHullPt p;
        p.x = X.x - V.x;
        p.y = X.y - V.y;
        p.w = gdt_dist2_64(p.x, p.y);
        return p;
    };
    const GdtHullPt c = pt(k), a = pt(lst[i]);
    // (the list stays short enough for the row table; the first entry stays
    // the nearest; and the triangle that this closes is no sliver, which every
    // other routine leaves uncertified)
    h.bad |= h.n + 1 > GDT_HULL_RING || c.w <= h.w0 ||
             !(gdt_hull_cross(a, c) > 1e-6 * (fabs(a.x * c.y) + fabs(a.y * c.x)));
    if (h.bad) {
        h.open = 0;
        return;
    }
    for (int q = h.n; q > i + 1; --q) lst[q] = lst[q - 1];
    lst[i + 1] = (gdt_u16a)k;
    ++h.n;
    const uint32_t low = (1u << (i + 1)) - 1u;
    h.open = (h.open & low & ~(1u << i)) | ((h.open & ~low) << 1) | (1u << (i + 1));
    auto convex = [&](const GdtHullPt& a, const GdtHullPt& b, const GdtHullPt& d) {
        const double ab = gdt_hull_cross(a, b), bd = gdt_hull_cross(b, d);
        const double P = gdt_hull_p(a, b, d, ab, gdt_hull_cross(a, d), bd);
        h.bad |= P == 0.;
        return ab > 0. && bd > 0. && P > 0.;
    };
    // entry at position j goes; its two triangles become one, open
    auto drop = [&](int j) {
        for (int q = j; q + 1 < h.n; ++q) lst[q] = lst[q + 1];
        --h.n;
        const uint32_t keep = (1u << j) - 1u;
        h.open = (h.open & keep) | ((h.open >> 1) & ~keep) | (1u << (j - 1));
    };
    int at = i + 1;
    while (at + 1 < h.n && !h.bad) {        // after it (the first entry is not dropped)
        const GdtHullPt b = pt(lst[at + 1]), d = pt(lst[at + 2 < h.n ? at + 2 : 0]);
        if (convex(c, b, d)) break;
        drop(at + 1);
    }
    while (at - 1 > 0 && !h.bad) {          // before it
        const GdtHullPt b = pt(lst[at - 1]), d = pt(lst[at - 2]);
        if (convex(d, b, c)) break;
        drop(at - 1);
        --at;
    }
    // the first entry, between the last and the second
    h.bad |= h.n < 3;
    if (!h.bad && !convex(pt(lst[h.n - 1]), pt(lst[0]), pt(lst[1]))) h.bad = true;
    if (h.bad) h.open = 0;
}

// Part 3 for one point, triangle after triangle.
template <bool GEN>
GDT_HD inline void gdt_hull_close(const GdtSet& S, const GdtTileLds& L,
                                  int iv, int c0, uint32_t* words, GdtHull& h, unsigned& npred)
{
    for (int round = 0; h.open != 0; ++round) {
        if (round >= GDT_HULL_ROUNDS) {
            h.bad = true;
            h.open = 0;
            break;
        }
        const int i = __builtin_ctz(h.open);
        const int ka = gdt_hull_entry(words, i), kb = gdt_hull_entry(words, i + 1 < h.n ? i + 1 : 0);
        const int k = gdt_hull_probe<GEN>(S, L, iv, c0, h.lv, ka, kb, words + GDT_HULL_TBL, 0,
                                          1, npred);
        h.open &= h.open - 1u;
        if (k == HULL_FAIL) {
            h.bad = true;
            h.open = 0;
        } else if (k >= 0) {
            gdt_hull_insert(L, iv, words, h, i, k);
        }
    }
}

// A point with open triangles, kept until a wave's worth of them is there.
// Word 1 is nonzero once the record is whole.
#define GDT_HULL_REC (2 + GDT_HULL_RING / 2)
GDT_HD inline void gdt_hull_save(const GdtHull& h, int iv, int c0, const uint32_t* words,
                                 uint32_t* rec)
{
    rec[0] = (uint32_t)iv | ((uint32_t)c0 << 16);
    for (int q = 0; q < GDT_HULL_RING / 2; ++q) rec[2 + q] = words[q];
#if defined(__HIPCC__)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __hip_atomic_store(rec + 1, h.open | ((uint32_t)h.n << 16) | ((uint32_t)h.lv << 24),
                       __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
#else
    rec[1] = h.open | ((uint32_t)h.n << 16) | ((uint32_t)h.lv << 24);
#endif
}
GDT_HD inline void gdt_hull_load(const GdtTileLds& L, const uint32_t* rec, GdtHull& h, int& iv,
                                 int& c0, uint32_t* words)
{
    iv = (int)(rec[0] & 0xffffu);
    c0 = (int)(rec[0] >> 16);
    h.open = rec[1] & 0xffffu;
    h.n = (int)(rec[1] >> 16) & 255;
    h.lv = (int)(rec[1] >> 24);
    h.bad = false;
    for (int q = 0; q < GDT_HULL_RING / 2; ++q) words[q] = rec[2 + q];
    const gdt_d2 V = L.X64[iv], X = L.X64[gdt_hull_entry(words, 0)];
    h.w0 = gdt_dist2_64(X.x - V.x, X.y - V.y);
}

#if defined(__HIPCC__)
// Part 3 for the points of a wave, GDT_HULL_W lanes per open triangle (1M-point
// kernel 350 us with two, 575 with one, 358 with four): up to two
// triangles of each lane at a time go to groups of lanes, which each scan a
// part of every row and agree on the first of their finds; the triangles' lanes
// then put those in, each lane's in the order that gdt_hull_close takes them, so that
// its row does not depend on the points that share the wave.  Every lane of the wave calls it (open = 0 where it has no
// point).  wave_words: the words of the wave's first lane; q: the wave's
// 2 GDT_HULL_GROUPS words.
#define GDT_HULL_W 2
#define GDT_HULL_GROUPS (64 / GDT_HULL_W)
template <bool GEN>
__device__ inline void gdt_hull_close_wave(const GdtSet& S, const GdtTileLds& L, int iv, int c0,
                                           uint32_t* wave_words, uint32_t* q, GdtHull& h,
                                           unsigned& npred)
{
    const int lane = (int)(threadIdx.x & 63);
    uint32_t* words = wave_words + GDT_HULL_WORDS * lane;
    const unsigned long long below = (1ull << lane) - 1ull;
    auto sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (int taken = 0;;) {
        if (taken >= GDT_HULL_ROUNDS && h.open != 0) {
            h.bad = true;
            h.open = 0;
        }
        const unsigned long long m1 = __ballot(h.open != 0);
        if (m1 == 0) break;
        const uint32_t rest = h.open & (h.open - 1u);
        const unsigned long long m2 = __ballot(rest != 0);
        const int i1 = h.open ? __builtin_ctz(h.open) : 0, i2 = rest ? __builtin_ctz(rest) : 0;
        const int p1 = __popcll(m1 & below), p2 = __popcll(m1) + __popcll(m2 & below);
        const int total = min(GDT_HULL_GROUPS, __popcll(m1) + __popcll(m2));
        const bool first = h.open != 0 && p1 < GDT_HULL_GROUPS;
        const bool second = rest != 0 && p2 < GDT_HULL_GROUPS;
        if (first) q[p1] = (uint32_t)(lane | (i1 << 6));
        if (second) q[p2] = (uint32_t)(lane | (i2 << 6));
        sync();
        const int g = lane / GDT_HULL_W, sub = lane & (GDT_HULL_W - 1);
        const uint32_t e = g < total ? q[g] : (uint32_t)lane;
        const int o = (int)(e & 63u), i = (int)(e >> 6);
        // the triangle's point: entry, window cell, block level, list length
        static_assert(GDT_WIN_MAXPTS <= 4096 && GDT_WIN_CELLS <= 2048, "a point's fields");
        const int po = __shfl(iv | (c0 << 12) | (h.lv << 23) | (h.n << 25), o, 64);
        int k = HULL_NONE, v = 0, ka = 0;
        if (g < total) {
            const uint32_t* ow = wave_words + GDT_HULL_WORDS * o;
            const int n = po >> 25;
            v = po & 4095;
            ka = gdt_hull_entry(ow, i);
            const int kb = gdt_hull_entry(ow, i + 1 < n ? i + 1 : 0);
            k = gdt_hull_probe<GEN>(S, L, v, (po >> 12) & 2047, (po >> 23) & 3, ka, kb,
                                    words + GDT_HULL_TBL, sub, GDT_HULL_W, npred);
        }
#pragma unroll
        for (int x = 1; x < GDT_HULL_W; x <<= 1) {
            const int pk = __shfl_xor(k, x, 64);
            int win = k;
            if (k == HULL_FAIL || pk == HULL_FAIL) {
                win = HULL_FAIL;
            } else if (k < 0) {
                win = pk;
            } else if (pk >= 0 && pk != k) {
                const gdt_d2 V = L.X64[v], A = L.X64[ka], B = L.X64[k], C = L.X64[pk];
                const GdtHullPt a = {A.x - V.x, A.y - V.y, gdt_dist2_64(A.x - V.x, A.y - V.y)};
                const GdtHullPt b = {B.x - V.x, B.y - V.y, gdt_dist2_64(B.x - V.x, B.y - V.y)};
                const GdtHullPt c = {C.x - V.x, C.y - V.y, gdt_dist2_64(C.x - V.x, C.y - V.y)};
                const double P = gdt_hull_p(a, b, c, gdt_hull_cross(a, b), gdt_hull_cross(a, c),
                                            gdt_hull_cross(b, c));
                win = P < 0. ? pk : (P == 0. ? HULL_FAIL : k);
            }
            k = __shfl(win, lane & ~(2 * x - 1), 64);   // (the lower lane's choice)
        }
        if (g < total && sub == 0) q[GDT_HULL_GROUPS + g] = (uint32_t)k;
        sync();
        // the triangle's lane: what was found goes into its list (a second
        // triangle's find then waits for the next round)
        auto take = [&](int at, int idx) {
            int r = (int)q[GDT_HULL_GROUPS + at];
            if (r == HULL_FAIL) {       // leaving the window: by this lane alone
                const int kn = gdt_hull_entry(words, idx + 1 < h.n ? idx + 1 : 0);
                r = gdt_hull_probe<GEN>(S, L, iv, c0, h.lv, gdt_hull_entry(words, idx), kn,
                                        words + GDT_HULL_TBL, 0, 1, npred);
            }
            ++taken;
            h.open &= ~(1u << idx);
            if (r == HULL_FAIL) {
                h.bad = true;
                h.open = 0;
            } else if (r >= 0) {
                gdt_hull_insert(L, iv, words, h, idx, r);
            }
            return r == HULL_NONE;
        };
        if (first && take(p1, i1) && second && taken < GDT_HULL_ROUNDS) take(p2, i2);
        sync();
    }
}
#endif
