// The tile routines (gdt_tile.h) against the per-point routines, for every
// point of a set; points a tile routine hands on go to the wavefront routine (64
// emulated lanes), as on the device.
// Usage: tile_rows <points.bin> <n> <lx> <ly> <cell size>
//   the exact mode (GDT_EXACT: FP64 and double-double decisions inside their
//   error bounds) against gdt_one_ring_exact, and every seventh point's row
//   again by the wavefront routine;
// or     tile_rows <points.bin> <n> <x11> <x22> <cell size> <x12> <x21>
//   FP64 in a general box (lattice vectors as columns) against gdt_one_ring_f64.
// Prints: points, points handed on, rows that differ, error flags.
#include "gdt_tile.h"
#include "gdt_exact_wave.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

// The FP64 tile steps of a point in a general box.
static GdtRingResult general_ring(const GdtSet& S, const GdtTileWin& w, const GdtTileLds& L, int j,
                                  const GdtRingIO& io)
{
    GdtRingResult res = {0, 0, 0u, 0u};
    uint32_t tbl[6];
    GdtTileLane<double> st;
    gdt_tile_lane_init_gen(w, L, j, io, S, st);
    st.tbl = tbl;
    int rc = STEP_RUN;
    while (rc == STEP_RUN) rc = gdt_tile_step_f64<1, false, true>(S, L, io, st, res.npred);
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
    const double lx = std::atof(argv[3]), ly = std::atof(argv[4]), cell = std::atof(argv[5]);
    std::vector<gdt_d2> xy((size_t)n);
    FILE* f = std::fopen(argv[1], "rb");
    if (!f || std::fread(xy.data(), sizeof(gdt_d2), (size_t)n, f) != (size_t)n) return 3;
    std::fclose(f);
    const double box[4] = {lx, general ? std::atof(argv[6]) : 0., general ? std::atof(argv[7]) : 0.,
                           ly};
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
    int handed = 0, differ = 0, err = 0;
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
            const GdtRingResult want =
                general ? gdt_one_ring_f64(S, j, io) : gdt_one_ring_exact(S, j, io);
            io.nbrs = rows[0].data();
            GdtRingResult got = {0, ERR_DEFER, 0u, 0u};
            if (fits && general) got = general_ring(S, w, L, j, io);
            else if (fits) got = gdt_tile_ring<GDT_EXACT>(S, w, L, j, io);
            const bool on = (got.err & ERR_DEFER) != 0;
            handed += on;
            if (on && general) got = gdt_wave_ring(S, j, io, wave, true);
            else if (on || (!general && j % 7 == 0)) got = gdt_wave_ring_exact(S, j, io, wave, true);
            err |= got.err;
            bool same = got.count == want.count && got.err == want.err;
            for (int m = 0; same && m < want.count && m < stride; ++m)
                same = rows[0][(size_t)perm[j] * stride + m] == rows[1][(size_t)perm[j] * stride + m];
            differ += same ? 0 : 1;
        }
    }
    std::printf("%d %d %d %d\n", n, handed, differ, err);
    return 0;
}
