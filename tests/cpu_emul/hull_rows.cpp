// The hull routine of the LDS tile kernels (gdt_hull.h) against the per-point
// FP64 routine, for every point of a set; points it leaves to the steps take
// them (gdt_tile.h), points those hand on the wavefront routine.
// Usage: hull_rows <points.bin> <n> <x11> <x22> <cell size> [<x12> <x21>]
// Prints: points, points left to the steps, rows that differ, error flags.
#include "gdt_hull.h"
#include "gdt_wave.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

template <bool GEN>
static GdtRingResult ring(const GdtSet& S, const GdtTileWin& w, const GdtTileLds& L, int j,
                          const GdtRingIO& io, int& left)
{
    GdtRingResult res = {0, 0, 0u, 0u};
    uint32_t words[GDT_HULL_WORDS + 1];
    GdtTileLane<double> st;
    gdt_tile_lane_init_gen(w, L, j, io, S, st);
    GdtHull h;
    gdt_hull_build<GEN>(S, L, st, words, h, res.npred);
    if (h.open != 0) {
        // as a block does: the list goes into a record, another lane closes it
        uint32_t rec[GDT_HULL_REC];
        int iv = -1, c0 = -1;
        gdt_hull_save(h, st.iv, st.c0, words, rec);
        for (uint32_t& w : words) w = 0xdeadbeefu;
        h = GdtHull{};
        gdt_hull_load(L, rec, h, iv, c0, words);
        gdt_hull_close<GEN>(S, L, iv, c0, words, h, res.npred);
    }
    if (!h.bad) {
        for (int i = 0; i < h.n && i < io.stride; ++i) st.row[i] = L.orig[gdt_hull_entry(words, i)];
        res.count = h.n;
        return res;
    }
    ++left;
    st.tbl = words + GDT_HULL_TBL;
    int rc = STEP_RUN;
    while (rc == STEP_RUN) rc = gdt_tile_step_f64<1, false, GEN>(S, L, io, st, res.npred);
    res.count = st.count;
    if (rc == STEP_DEFER) res.err = ERR_DEFER;
    if (rc == STEP_NOCLOSE) res.err = ERR_NOCLOSE;
    return res;
}

int main(int argc, char** argv)
{
    if (argc != 6 && argc != 8) return 2;
    const bool general = argc == 8;
    const int n = std::atoi(argv[2]), stride = 32;
    const double cell = std::atof(argv[5]);
    const double box[4] = {std::atof(argv[3]), general ? std::atof(argv[6]) : 0.,
                           general ? std::atof(argv[7]) : 0., std::atof(argv[4])};
    std::vector<gdt_d2> xy((size_t)n);
    FILE* f = std::fopen(argv[1], "rb");
    if (!f || std::fread(xy.data(), sizeof(gdt_d2), (size_t)n, f) != (size_t)n) return 3;
    std::fclose(f);
    const GdtSet S = gdt_make_set_box(0, n, 0, box, cell, 1);
    std::vector<uint32_t> cstart((size_t)S.nkeys + 1, 0u), scell((size_t)n);
    std::vector<int> key((size_t)n), perm((size_t)n);
    std::vector<gdt_d2> off((size_t)n);
    for (int i = 0; i < n; ++i) {
        int cx, cy;
        double ox, oy;
        gdt_bin_point(S, xy[i].x, xy[i].y, cx, cy, ox, oy);
        key[i] = gdt_cell_key(S, cx, cy);
        ++cstart[(size_t)key[i] + 1];
    }
    for (int k = 0; k < S.nkeys; ++k) cstart[(size_t)k + 1] += cstart[(size_t)k];
    std::vector<uint32_t> at(cstart.begin(), cstart.end() - 1);
    for (int i = 0; i < n; ++i) {
        const uint32_t j = at[(size_t)key[i]]++;
        int cx, cy;
        perm[j] = i;
        gdt_bin_point(S, xy[i].x, xy[i].y, cx, cy, off[j].x, off[j].y);
        scell[j] = (uint32_t)cx | ((uint32_t)cy << 16);
    }
    std::vector<int> rows[2];
    for (auto& r : rows) r.assign((size_t)n * stride, -1);
    GdtRingIO io = {};
    io.cstart = cstart.data(); io.perm = perm.data(); io.off64 = off.data();
    io.scell = scell.data(); io.stride = stride; io.xy = xy.data();
    std::vector<uint32_t> cs(GDT_WIN_CELLS + 1), cnt(GDT_WIN_CELLS);
    std::vector<int> gs(GDT_WIN_CELLS), orig(GDT_WIN_MAXPTS);
    std::vector<gdt_d2> X64(GDT_WIN_MAXPTS + 1);
    GdtTileLds L = {cs.data(), gs.data(), X64.data(), nullptr, orig.data()};
    GdtWaveHost wave;
    int left = 0, differ = 0, err = 0;
    for (int t = 0; t < S.nkeys / GDT_TILE_CELLS; ++t) {
        const GdtTileWin w = gdt_tile_window(S, t);
        uint32_t run = 0;
        for (int c = 0; c < GDT_WIN_CELLS; ++c) {
            gdt_tile_count(S, w, c, io.cstart, gs[c], cnt[c]);
            cs[c] = run;
            run += cnt[c];
        }
        cs[GDT_WIN_CELLS] = run;
        const bool fits = run <= GDT_WIN_MAXPTS && S.rmax >= GDT_SCAN;
        for (int c = 0; c < GDT_WIN_CELLS && fits; ++c)
            for (uint32_t k = 0; k < cnt[c]; ++k) {
                const int fx = c % GDT_WIN - GDT_FRAME, fy = c / GDT_WIN - GDT_FRAME;
                L.X64[cs[c] + k] = gdt_frame64_gen(S, fx, fy, io.off64[gs[c] + (int)k]);
                L.orig[cs[c] + k] = io.perm[gs[c] + (int)k];
            }
        const int k0 = t * GDT_TILE_CELLS;
        for (int j = (int)cstart[k0]; j < (int)cstart[k0 + GDT_TILE_CELLS]; ++j) {
            io.nbrs = rows[1].data();
            GdtRingResult want = gdt_one_ring_f64(S, j, io);
            if (want.err & ERR_SEARCH) want = gdt_wave_ring(S, j, io, wave, true);
            io.nbrs = rows[0].data();
            GdtRingResult got = {0, ERR_DEFER, 0u, 0u};
            if (fits)
                got = general ? ring<true>(S, w, L, j, io, left) : ring<false>(S, w, L, j, io, left);
            if (got.err & ERR_DEFER) got = gdt_wave_ring(S, j, io, wave, true);
            err |= got.err;
            bool same = got.count == want.count && got.err == want.err;
            for (int q = 0; same && q < want.count && q < stride; ++q)
                same = rows[0][(size_t)perm[j] * stride + q] == rows[1][(size_t)perm[j] * stride + q];
            differ += same ? 0 : 1;
        }
    }
    std::printf("%d %d %d %d\n", n, left, differ, err);
    return 0;
}
