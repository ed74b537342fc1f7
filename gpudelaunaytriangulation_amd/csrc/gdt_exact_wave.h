// gdt_exact_wave.h -- gdt_one_ring_exact (gdt_exact_ring.h) with a wavefront
// per point (host/device): the same searches, decisions, stops and errors,
// the cells of a pass dealt to the 64 lanes and the lane bests reduced (a
// tree over the exact total order on the candidates keeps the sequential
// scan's choice).  For the points the exact mode's tile and star kernels hand
// on: a handful on random input, bound by one point's chain of dependent
// passes.  Measured on 2^18 random points (a few handed on): 111 us for the
// kernel, 1,131 us with one lane per point.
#pragma once

#include "gdt_exact_ring.h"
#include "gdt_wave.h"

// Rings of cells a pass adds at most.
#define GDT_XWAVE_GROW 8

// The comparisons of one point's searches; `overflow` is this lane's.
struct GdtXWave {
    const GdtSet& S;
    const GdtRingIO& io;
    int j;
    gdt_d2 pv;
    double L;
    GdtXCtx xc;

    GDT_HD GdtDDVec dd(const GdtWaveBest& c) const
    {
        return gdt_dd_disp(pv, io.xy[io.perm[c.k]], S.lx, S.ly, c.x, c.y);
    }
    GDT_HD void exact(const GdtWaveBest& c, GdtXVec& X)
    {
        gdt_x_disp(pv, io.xy[io.perm[c.k]], S.lx, S.ly, c.x, c.y, X.x, X.y, xc);
    }
    GDT_HD static double mag(const GdtWaveBest& c) { return GDT_FMAX(fabs(c.x), fabs(c.y)); }

    // c is nearer than b (exact ties: the lower caller index)
    GDT_HD bool closer(const GdtWaveBest& c, const GdtWaveBest& b)
    {
        const double mc = mag(c), mb = mag(b);
        const double tol = gdt_x_tol2(gdt_x_err(L, mc), mc) + gdt_x_tol2(gdt_x_err(L, mb), mb);
        if (c.d2 < b.d2 - tol) return true;
        if (c.d2 > b.d2 + tol) return false;
        const double M = GDT_FMAX(mc, mb);
        int s = gdt_dd_sign(gdt_dd_dist_cmp(dd(c), dd(b)), 2. * gdt_dd_tol2(gdt_dd_err(L, M), M));
        if (s == 0) {
            GdtXVec C, B;
            exact(c, C);
            exact(b, B);
            s = gdt_x_dist_cmp(C, B, xc);
        }
        return s < 0 || (s == 0 && gdt_nn_tie(io.perm[c.k], io.perm[b.k]));
    }
    // c is strictly left of v->a
    GDT_HD bool left(const GdtWaveBest& a, const GdtWaveBest& c)
    {
        const double O = gdt_orient64(a.x, a.y, c.x, c.y);
        const double M = GDT_FMAX(mag(a), mag(c));
        const double tol = gdt_x_tol2(gdt_x_err(L, M), M);
        if (O > tol) return true;
        if (O < -tol) return false;
        int s = gdt_dd_sign(gdt_dd_orient(dd(a), dd(c)), gdt_dd_tol2(gdt_dd_err(L, M), M));
        if (s == 0) {
            GdtXVec A, C;
            exact(a, A);
            exact(c, C);
            s = gdt_x_orient(A, C, xc);
        }
        return s > 0;
    }
    // c (left of v->a) lies inside the circle through v, a and b
    GDT_HD bool inside(const GdtWaveBest& a, const GdtWaveBest& b, const GdtWaveBest& c)
    {
        const double P = gdt_incircle64(gdt_circ64(a.x, a.y, b.x, b.y), c.x, c.y);
        const double M = GDT_FMAX(GDT_FMAX(mag(a), mag(b)), mag(c));
        const double tol = gdt_x_tol4(gdt_x_err(L, M), M);
        if (P < -tol) return true;
        if (P > tol) return false;
        int s = gdt_dd_sign(gdt_dd_incircle(dd(a), dd(b), dd(c)), gdt_dd_tol4(gdt_dd_err(L, M), M));
        if (s != 0) return s < 0;
        GdtXVec A, B, C;
        exact(a, A);
        exact(b, B);
        exact(c, C);
        s = gdt_x_incircle(A, B, C, xc);
        return s < 0 || (s == 0 && gdt_x_incircle_tie(io.perm[j], io.perm[a.k], io.perm[b.k],
                                                      io.perm[c.k], A, B, C, xc));
    }
};

template <class W>
GDT_HD inline GdtRingResult gdt_wave_ring_exact(const GdtSet& S, int j, const GdtRingIO& io, W& w,
                                                bool lead)
{
    GdtRingResult res = {0, 0, 0u, 0u};
    const uint32_t pc = io.scell[j];
    const int cx = (int)(pc & 0xffffu), cy = (int)(pc >> 16);
    const gdt_d2 ov = io.off64[j];
    const double covb = gdt_cover0(S, ov.x, ov.y), bsmin = S.hmin;
    const size_t row = (size_t)io.perm[j] * (size_t)io.stride;
    GdtXWave X = {S, io, j, io.xy[io.perm[j]], S.lx > S.ly ? S.lx : S.ly, {false}};
    if (S.general || !(fabs(X.pv.x) <= 4. * S.lx && fabs(X.pv.y) <= 4. * S.ly)) {
        res.err = ERR_RANGE;
        return res;
    }
    unsigned npred = 0;
    GdtWaveBest a = gdt_wave_none(), g;
    // Nearest neighbour (a.k < 0) or successor of a: passes over the cells of
    // [-h,h]^2 outside the previous square, from h = 2 on (the smaller
    // squares' stops are met there too, with the same best).
    auto search = [&]() -> bool {
        const bool wrap = a.k >= 0;
        g = gdt_wave_none();
        auto better = [&](const GdtWaveBest& b, const GdtWaveBest& c) {
            if (c.k < 0 || c.k == b.k) return false;
            if (b.k < 0) return true;
            return wrap ? X.inside(a, b, c) : X.closer(c, b);
        };
        auto pass = [&](int x0, int x1, int y0, int y1, int hole) {
            const int nx = x1 - x0 + 1, ncell = nx * (y1 - y0 + 1);
            auto lane_fn = [&](int lane, GdtWaveBest& m) {
                for (int q = lane; q < ncell; q += GDT_WAVE) {
                    const int dx = x0 + q % nx, dy = y0 + q / nx;
                    if (dx >= -hole && dx <= hole && dy >= -hole && dy <= hole) continue;
                    const int x = gdt_wrap(cx + dx, S.xsize), y = gdt_wrap(cy + dy, S.ysize);
                    const int key = S.c0 + gdt_cell_key(S, x, y);
                    const uint32_t b = io.cstart[key], e = io.cstart[key + 1];
                    const double bx = gdt_cbase_x(S, dx, dy, ov.x), by = gdt_cbase_y(S, dx, dy, ov.y);
                    for (uint32_t k = b; k < e; ++k) {
                        if ((int)k == j || (int)k == a.k) continue;
                        const gdt_d2 o = io.off64[k];
                        GdtWaveBest c;
                        c.k = (int)k;
                        c.x = gdt_disp64(bx, o.x);
                        c.y = gdt_disp64(by, o.y);
                        c.d2 = gdt_dist2_64(c.x, c.y);
                        ++npred;
                        if (wrap && !X.left(a, c)) continue;
                        if (better(m, c)) m = c;
                    }
                }
            };
            g = w.ring_by(g, lane_fn, better);
        };
        // the per-point routine's stop after the rings 0..h
        auto done = [&](int h) {
            if (!wrap) {
                const double cov = (double)h * bsmin + covb - 4. * gdt_x_err(X.L, (double)(h + 1) * bsmin);
                return cov > 0. && g.d2 <= cov * cov * (1.0 - 1e-9);
            }
            const double cov = (double)h * bsmin + covb;
            const Circ64 K = gdt_circ64(a.x, a.y, g.x, g.y);
            const double k0min = 1e-6 * (fabs(a.x * g.y) + fabs(a.y * g.x));
            return K.k0 > k0min && cov > 0. &&
                   K.kx * K.kx + K.ky * K.ky <= cov * cov * (K.k0 * K.k0) * (1.0 - 1e-6);
        };
        // The square [-h,h]^2 first.  A search whose best would be certified
        // within the search radius goes to the first square that certifies
        // it in one pass (a later best's circle is smaller on the left of v->a,
        // but may stop it only later: the test is repeated); else ring by ring.
        int h = S.rmax < 2 ? S.rmax : 2;
        pass(-h, h, -h, h, -1);
        for (;;) {
            if (g.k >= 0 && done(h)) return true;
            if (h >= S.rmax) return false;
            int to = h + 1;
            if (g.k >= 0) {
                while (to < S.rmax && to < h + GDT_XWAVE_GROW && !done(to)) ++to;
            }
            pass(-to, to, -to, to, h);
            h = to;
        }
    };
    int nn = -1, count = 0;
    for (;;) {
        if (!search()) {
            res.err |= g.k < 0 ? ERR_NONEIGHBOUR : ERR_SEARCH;
            break;
        }
        if (nn >= 0 && g.k == nn) break;
        if (nn < 0) nn = g.k;
        a = g;
        if (lead && count < io.stride) io.nbrs[row + count] = io.perm[a.k];
        ++count;
        if (count > GDT_HARD_CAP) { res.err |= ERR_NOCLOSE; break; }
    }
    if (X.xc.overflow) res.err |= ERR_NONEIGHBOUR;      // (this lane's: the caller joins them)
    res.count = count;
    res.npred = npred;
    return res;
}
