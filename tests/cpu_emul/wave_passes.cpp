// The FP64 wavefront routine (gdt_wave.h) with its passes counted (those of a
// search that has a candidate), against the per-point routine, for every point
// of a set.
// Usage: wave_passes <points.bin> <n> <x11> <x22> <cell size> [<x12> <x21>]
// Prints: points, rows that differ, most passes to a ring entry (a point's average).
#include "gdt_wave.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

struct CountingWave : GdtWaveHost {
    int passes = 0;
    template <bool TIES, class Fn>
    GdtWaveBest ring(const GdtWaveBest& start, bool wrap, double ax, double ay, GdtTieIds& t, Fn& fn)
    {
        passes += start.k >= 0;
        return GdtWaveHost::ring<TIES>(start, wrap, ax, ay, t, fn);
    }
};

int main(int argc, char** argv)
{
    if (argc != 6 && argc != 8) return 2;
    const bool general = argc == 8;
    const int n = std::atoi(argv[2]), stride = 64;
    const double box[4] = {std::atof(argv[3]), general ? std::atof(argv[6]) : 0.,
                           general ? std::atof(argv[7]) : 0., std::atof(argv[4])};
    std::vector<gdt_d2> xy((size_t)n);
    FILE* f = std::fopen(argv[1], "rb");
    if (!f || std::fread(xy.data(), sizeof(gdt_d2), (size_t)n, f) != (size_t)n) return 3;
    std::fclose(f);
    const GdtSet S = gdt_make_set_box(0, n, 0, box, std::atof(argv[5]), 0);
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
    int differ = 0, most = 0;
    for (int j = 0; j < n; ++j) {
        io.nbrs = rows[1].data();
        const GdtRingResult want = gdt_one_ring_f64(S, j, io);
        io.nbrs = rows[0].data();
        CountingWave w;
        const GdtRingResult got = gdt_wave_ring(S, j, io, w, true);
        if (got.count > 0) most = std::max(most, w.passes / (got.count + 1));
        bool same = got.count == want.count && (got.err != 0) == (want.err != 0);
        for (int q = 0; same && q < want.count && q < stride; ++q)
            same = rows[0][(size_t)perm[j] * stride + q] == rows[1][(size_t)perm[j] * stride + q];
        differ += same ? 0 : 1;
    }
    std::printf("%d %d %d\n", n, differ, most);
    return 0;
}
