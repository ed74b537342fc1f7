// tile.hip -- the LDS-staged one-ring kernel (one block per tile of cells).
//
// Compiled once per supported tile edge: GDT_TILE_SHIFT (4: 16x16 cells, 5:
// 32x32) and the window's LDS point budget GDT_WIN_MAXPTS come from the
// compile line, and everything here lives in namespace ts<shift>, so both
// builds link into one library (gdt_kernels.h declares both launchers).
// Replaces gpu_voronoi_calc_global_kernel + gpu_get_neighbors_global_kernel
// (DelaunayGPU.cu:649-675, 981-1006) and their masked repair variants
// (DelaunayGPU.cu:611-640, 945-975).
#include "gdt_hull.h"
#include "gdt_kernels.h"
#include "gdt_stage.h"
#include "gdt_wavedev.h"

#include <type_traits>

namespace GDT_TS_NS {

// k_one_ring_tile: one block per tile (GDT_TILE x GDT_TILE cells, this file's
// compiled tile edge): stage the tile window in LDS, then the lanes advance the
// tile's points one search step at a time.  With `flags` null the tile's points
// are all its slots [T0, T1); with `flags` (a caller-order array, flagged >= 0)
// they are the tile's flagged slots, which the block gathers first into a bit
// mask in LDS (status[ST_NFLAGGED] += their count).  A tile with none exits
// before staging.  The points of a window that does not fit the LDS budget, or
// of a grid too small for the scan block, and points with a step whose circle
// leaves the window, are appended to `defer` and handled by k_one_ring_deferred
// in the next launch.  With W = 2 or 4 (FP64) neighbouring lanes share each
// point, each scanning its part of every row (flags leave most lanes of a
// block without a point otherwise, and a small grid leaves most of the chip
// idle; the launcher takes W from the caller).  One lane per point, in FP64 or
// FP32-filtered, is k_one_ring_hull's.  GEN: sets in general boxes (gdt_tile_search_f64).
// PREC = GDT_EXACT: the FP64 steps with every decision certified
// (gdt_tile_search_f64, CERT), bound as they are by the lanes' chains of steps;
// all its deferred points go to the next launch, where a wavefront per point
// takes the expansions.  Kernel times against the per-point exact kernel: 2^18
// random points 290 us (2,427 us), 65,536 points of a square lattice off by
// 1e-13 207 us + 147 us deferred (4,171 us).

// The tile's flagged slots (flags mode): slot T0 + 64 w + b is flagged when bit
// b of mask[w] is set; pre[w] = flagged slots before word w.
struct TileFlags {
    const unsigned long long* mask;
    const uint32_t* pre;
    int nw;     // words
};

// Slot of the q-th flagged slot (q below the tile's count).
__device__ inline int tile_flagged_slot(const TileFlags& f, int T0, int q)
{
    int lo = 0, hi = f.nw - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if ((int)f.pre[mid] <= q) lo = mid; else hi = mid - 1;
    }
    unsigned long long m = f.mask[lo];
    for (int r = q - (int)f.pre[lo]; r > 0; --r) m &= m - 1ull;
    return T0 + 64 * lo + __ffsll((long long)m) - 1;
}

// Prefix counts pre[0..nw] of a mask's words (nw <= 64), by the first wave;
// returns the total (every thread calls it; ends with a barrier).
__device__ inline int tile_mask_prefix(const TileFlags& f, uint32_t* pre)
{
    const int tid = threadIdx.x;
    if (tid < 64) {
        uint32_t x = tid < f.nw ? (uint32_t)__popcll(f.mask[tid]) : 0u;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(x, d, 64);
            if (tid >= d) x += y;
        }
        if (tid < f.nw) pre[tid + 1] = x;
        if (tid == 0) pre[0] = 0u;
    }
    __syncthreads();
    return (int)pre[f.nw];
}

// Gathers the tile's flagged slots (flags[caller index] >= 0) into a bit mask and
// its prefix counts; returns their number (block-uniform, ends with a barrier).
__device__ inline int tile_gather_flags(const int* __restrict__ flags, const int* __restrict__ perm,
                                        int T0, int npt, unsigned long long* mask, uint32_t* pre,
                                        TileFlags& tf)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    tf.mask = mask;
    tf.pre = pre;
    tf.nw = (npt + 63) >> 6;
    for (int t0 = 0; t0 < 64 * tf.nw; t0 += nt) {
        const int t = t0 + tid;
        const bool f = t < npt && flags[perm[T0 + t]] >= 0;
        const unsigned long long b = __ballot(f);
        if ((tid & 63) == 0 && (t >> 6) < tf.nw) mask[t >> 6] = b;
    }
    __syncthreads();
    return tile_mask_prefix(tf, pre);
}

// The points a tile block deferred (their circle left the window): one
// wavefront each, read from global memory (gdt_wave_ring), by this block's waves while
// other blocks still run their tiles.  Built without the tie rule and the
// other box shape, which would cost the kernels' main loops registers: a point
// with an exact tie goes to k_one_ring_deferred.
template <bool GEN>
__device__ inline void tile_finish_deferred(const GdtSet& S, const GdtRingIO& io, const int* dlist,
                                            int ndl, int* __restrict__ counts,
                                            int* __restrict__ status, int* __restrict__ defer,
                                            unsigned& npred, unsigned& nsum, int& mx, int& er)
{
    if (ndl <= 0) return;
    const int tid = threadIdx.x, nt = blockDim.x;
    if (tid == 0) atomicAdd(&status[ST_NDEFER_TILE], ndl);
    GdtWaveDev wv;
    wv.lane = tid & 63;
    for (int t = tid >> 6; t < ndl; t += nt >> 6) {
        const int jd = dlist[t];
        const GdtRingResult r = gdt_wave_ring<false, GEN>(S, jd, io, wv, wv.lane == 0);
        npred += r.npred;
        if (r.err & ERR_TIE) {
            if (wv.lane == 0) {
                const uint32_t pos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u);
                defer[pos] = jd;
            }
        } else if (wv.lane == 0) {
            counts[io.perm[jd]] = r.count;
            mx = max(mx, r.count);
            er |= r.err;
            nsum += (unsigned)r.count;
        }
    }
}

// Block totals of a ring kernel (every thread calls it): one set of atomics
// per block, not per wave.
__device__ inline void ring_block_totals(int mx, int er, unsigned npred, unsigned nfb,
                                         unsigned nsum, int* status, unsigned long long* counters)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    mx = wave_max_i32(mx);
    er = wave_or_i32(er);
    npred = wave_sum_u32(npred);
    nfb = wave_sum_u32(nfb);
    nsum = wave_sum_u32(nsum);
    __shared__ unsigned s_red[5][16];
    if ((tid & 63) == 0) {
        const int w = tid >> 6;
        s_red[0][w] = (unsigned)mx;
        s_red[1][w] = (unsigned)er;
        s_red[2][w] = npred;
        s_red[3][w] = nfb;
        s_red[4][w] = nsum;
    }
    __syncthreads();
    if (tid == 0) {
        unsigned long long bp = 0, bf = 0, bs = 0;
        int bm = 0, be = 0;
        for (int w = 0; w < (nt >> 6); ++w) {
            bm = max(bm, (int)s_red[0][w]);
            be |= (int)s_red[1][w];
            bp += s_red[2][w];
            bf += s_red[3][w];
            bs += s_red[4][w];
        }
        if (bm > 0) atomicMax(&status[ST_REQUIRED], bm);
        if (be) atomicOr(&status[ST_ERRFLAGS], be);
        if (bp) atomicAdd(&counters[CT_PRED], bp);
        if (bf) atomicAdd(&counters[CT_FALLBACK], bf);
        if (bs) atomicAdd(&counters[CT_NBRSUM], bs);
    }
}

template <int PREC, int W, bool GEN = false>
__global__ __launch_bounds__(PREC == GDT_EXACT ? GDT_XTILE_BLOCK : 1024) void k_one_ring_tile(const GdtSet* __restrict__ sets, const GdtChunk* __restrict__ tiles,
                     const int* __restrict__ flags, const int* __restrict__ halt,
                     GdtRingIO io, int* __restrict__ counts, int* __restrict__ status,
                     unsigned long long* __restrict__ counters, int* __restrict__ defer)
{
    __shared__ uint32_t s_cs[GDT_WIN_CELLS + 1];
    __shared__ gdt_d2 s_X64[GDT_WIN_MAXPTS + 1];     // (+1: read by the scan's last prefetch)
    __shared__ gdt_f2 s_X32[PREC == 32 ? GDT_WIN_MAXPTS + 1 : 1];
    __shared__ int s_orig[GDT_WIN_MAXPTS];
    __shared__ uint32_t s_wsum[16];
    __shared__ int s_next;
    __shared__ int s_dlist[GDT_TILE_DEFER];
    __shared__ uint32_t s_dn;
    __shared__ unsigned long long s_fmask[GDT_WIN_MAXPTS / 64];
    __shared__ uint32_t s_fpre[GDT_WIN_MAXPTS / 64 + 1];
    extern __shared__ uint32_t s_tbl[];     // [5 * blockDim + 1] the lanes' row tables

    const GdtChunk ch = tiles[blockIdx.x];
    const GdtSet S = sets[ch.set];
    const GdtTileWin w = gdt_tile_window(S, ch.start);
    GdtTileLds L;
    L.cs = s_cs; L.gstart = nullptr; L.X64 = s_X64; L.X32 = s_X32; L.orig = s_orig;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int k0 = S.c0 + ch.start * GDT_TILE_CELLS;
    const int T0 = (int)io.cstart[k0], T1 = (int)io.cstart[k0 + GDT_TILE_CELLS];
    // the tile's items q in [Q0, Q1): point j = item(q)
    int Q0 = T0, Q1 = T1;
    TileFlags tf = {s_fmask, s_fpre, 0};
    if (flags) {
        if (halt && *halt) return;
        const int npt = T1 - T0;
        if (npt > GDT_WIN_MAXPTS) {
            // (more points than a window holds: the window cannot fit either)
            unsigned nf = 0;
            for (int q = T0 + tid; q < T1; q += nt)
                if (flags[io.perm[q]] >= 0) {
                    ++nf;
                    const uint32_t pos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u);
                    defer[pos] = q;
                }
            if (nf) atomicAdd(&status[ST_NFLAGGED], (int)nf);
            return;
        }
        Q0 = 0;
        Q1 = tile_gather_flags(flags, io.perm, T0, npt, s_fmask, s_fpre, tf);
        if (tid == 0 && Q1 > 0) atomicAdd(&status[ST_NFLAGGED], Q1);
    }
    auto item = [&](int q) { return flags ? tile_flagged_slot(tf, T0, q) : q; };
    if (Q0 >= Q1) return;    // block-uniform: nothing to do in this tile

    const bool fits = gdt_stage_window<PREC == 32, GEN>(S, w, io, L, s_wsum);

    if (!fits) {
        for (int q = Q0 + tid; q < Q1; q += nt) {
            const uint32_t pos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u);
            defer[pos] = item(q);
        }
        return;
    }
    // Lanes take points of the tile and advance them one search step per
    // iteration; a lane whose point is finished takes the next one, so a
    // wave's iterations track the total number of steps, not the longest ring.
    static_assert(W == 1 || W == 2 || (W == 4 && PREC == 64), "1, 2 or (FP64) 4 lanes per point");
    static_assert(!GEN || (PREC == 64 && W <= 2), "general boxes: FP64, one or two lanes");
    static_assert(PREC == 32 || PREC == 64 || PREC == GDT_EXACT, "a precision code");
    unsigned npred = 0, nfb = 0, nsum = 0;
    int mx = 0, er = 0;
    auto run = [&](auto lanes_each) {
        constexpr int V = decltype(lanes_each)::value;      // lanes per point
        if (tid == 0) {
            s_next = Q0 + nt / V;
            s_dn = 0u;
        }
        __syncthreads();
        using Real = typename std::conditional<PREC == 32, float, double>::type;
        GdtTileLane<Real> st;
        st.tbl = s_tbl + 5 * tid;
        const int sub = tid & (V - 1);      // the lane's part of its point's rows
        int q = Q0 + tid / V;
        bool have = q < Q1;
        int j = have ? item(q) : 0;
        auto lane_init = [&]() {
            if constexpr (GEN) gdt_tile_lane_init_gen(w, L, j, io, S, st);
            else gdt_tile_lane_init<Real>(w, L, j, io, S, st);
        };
        if (have) lane_init();
        while (__ballot(have) != 0) {
            if (have) {
                int rc;
                if constexpr (PREC == 32)
                    rc = gdt_tile_step_f32<V>(S, L, io, st, npred, nfb, sub);
                else
                    rc = gdt_tile_step_f64<V, PREC == GDT_EXACT, GEN>(S, L, io, st, npred, sub);
                // (both lanes of a pair end each step in the same state; the first reports)
                if (rc != STEP_RUN && sub == 0) {
                    if (rc == STEP_DEFER) {
                        // the block's own waves finish it after the tile (below)
                        // (the exact mode's go to the per-point routine)
                        const uint32_t dpos = PREC == GDT_EXACT ? GDT_TILE_DEFER : atomicAdd(&s_dn, 1u);
                        if (dpos < GDT_TILE_DEFER) {
                            s_dlist[dpos] = j;
                        } else {
                            const uint32_t pos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u);
                            defer[pos] = j;
                        }
                    } else {
                        counts[L.orig[st.iv]] = st.count;
                        mx = max(mx, st.count);
                        nsum += (unsigned)st.count;
                        if (rc == STEP_NOCLOSE) er |= ERR_NOCLOSE;
                    }
                }
                if (rc != STEP_RUN) {
                    if constexpr (V > 1) {
                        int qq = 0;
                        if (sub == 0) qq = atomicAdd(&s_next, 1);
                        q = __shfl(qq, (tid & 63) & ~(V - 1), 64);
                    } else {
                        q = atomicAdd(&s_next, 1);
                    }
                    have = q < Q1;
                    if (have) {
                        j = item(q);
                        lane_init();
                    }
                }
            }
        }
    };
    // A repair's four lanes per point are for the few points of a tile; where they
    // outnumber the block's groups of four, two lanes each take them in half as many
    // turns (test and repair of 65,536 points moved by 0.05, 143 of a tile's 256
    // flagged: 223 us, 244 with four lanes; by 0.01, 40 flagged: 176 with four, 198 with
    // two; the line at 64 or 85 flagged made no difference).
    if constexpr (W == 4) {
        if (flags && 4 * (Q1 - Q0) > nt) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 4>{});
    } else {
        run(std::integral_constant<int, W>{});
    }
    if constexpr (PREC != GDT_EXACT) {
        __syncthreads();
        tile_finish_deferred<GEN>(S, io, s_dlist, min((int)s_dn, GDT_TILE_DEFER), counts, status,
                                  defer, npred, nsum, mx, er);
    }
    ring_block_totals(mx, er, npred, nfb, nsum, status, counters);
}

// Words of a star lane's row table: one per cell row of the 7x7 block (the
// uniform scan reads no word beyond its rows; a step's own tables, at most
// five rows and the word read after them, fit in the first six).
#define STAR_TBL (2 * GDT_SCAN + 1)
// Points handed on that a star block keeps for one append (more go one by one).
#define STAR_HAND 256

// Whether two entries of the lanes' block (one each, kg; half its edge ph) are at the
// point's smallest distance as far as the exact mode's bounds tell.
__device__ inline bool star_nn_tie(const GdtSet& S, const GdtTileLds& L, const GdtRingIO& io,
                                   const GdtTileLane<double>& st, int kg, int ph)
{
    const bool here = kg >= 0 && kg != st.iv;
    const gdt_d2 X = L.X64[here ? kg : st.iv];
    const double x = X.x - st.vx, y = X.y - st.vy;
    const double d2 = here ? gdt_dist2_64(x, y) : 1e300;
    double least = d2;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) least = GDT_FMIN(least, __shfl_xor(least, o, 64));
    const double Lbox = GDT_FMAX(S.lx, S.ly), M = (double)(ph + 1) * GDT_FMAX(S.bsx, S.bsy);
    const bool near = here && d2 <= least + 2. * gdt_x_tol2(gdt_x_err(Lbox, M), M);
    const unsigned long long m = __ballot(near);
    if (m == 0ull || (m & (m - 1ull)) == 0ull) return false;
    // (against the first of them)
    const int first = __ffsll((long long)m) - 1;
    const gdt_d2 pv = io.xy[L.orig[st.iv]];
    GdtDDVec c = {{0., 0.}, {0., 0.}}, b;
    if (near) c = gdt_dd_disp(pv, io.xy[L.orig[kg]], S.lx, S.ly, x, y);
    b.x.h = __shfl(c.x.h, first, 64);
    b.x.l = __shfl(c.x.l, first, 64);
    b.y.h = __shfl(c.y.h, first, 64);
    b.y.l = __shfl(c.y.l, first, 64);
    const int s = gdt_dd_sign(gdt_dd_dist_cmp(c, b), 2. * gdt_dd_tol2(gdt_dd_err(Lbox, M), M));
    return __any(near && (int)(threadIdx.x & 63) != first && s == 0);
}

// One point by a wavefront (st: the point's state, the same in every lane, with
// the lane's own table of STAR_TBL words; k_one_ring_star describes it).  Returns
// STEP_DONE, STEP_NOCLOSE or STEP_DEFER, the row's length in count (CERT: tied,
// where a lane met a tie).
template <bool CERT, bool GEN>
__device__ inline int star_ring(const GdtSet& S, const GdtTileLds& L, const GdtRingIO& io,
                                GdtTileLane<double>& st, unsigned& npred, int& count, bool& tied)
{
    const int lane = (int)(threadIdx.x & 63);
    // the lanes' block, as one row table (every lane the same): the
    // (2 GDT_SCAN + 1)^2 cells when they hold at most 64 entries, else
    // the (2 GDT_SCAN0 + 1)^2 cells; and this lane's entry of it
    const GdtClip whole = {0.f, 0.f, 0};
    int ph = GDT_SCAN;
    int tot = (int)gdt_block_rows(L, st.c0, ph, whole, st.tbl);
    if (tot > 64) {
        ph = GDT_SCAN0;
        tot = (int)gdt_block_rows(L, st.c0, ph, whole, st.tbl);
    }
    int kg = -1;
    for (int acc = 0, r = 0; acc < tot; ++r) {      // (the table's non-empty rows)
        const uint32_t t = st.tbl[r];
        const int b = (int)(t & 0xffffu), n = (int)(t >> 16) - b;
        if (lane >= acc && lane < acc + n) kg = b + lane - acc;
        acc += n;
    }
    // (a block that holds too many for the lanes: lane 0's chain of steps is the
    // slower way with certified decisions, and in general boxes, whose clumps are
    // handed on)
    if ((CERT || GEN) && tot > 64) return STEP_DEFER;
    if constexpr (CERT) {
        // a point with two nearest neighbours, which the lanes' searches would
        // end at (every point of a square lattice), is handed on at once
        if (star_nn_tie(S, L, io, st, kg, ph)) {
            tied = true;
            return STEP_DEFER;
        }
    }
    int bk = -1, rc = STEP_DEFER;
    if (tot <= 64 && kg >= 0) {
        GdtTileLane<double> sl = st;
        if (kg != st.iv) {
            const gdt_d2 X = L.X64[kg];
            sl.ak = kg;
            sl.ax = X.x - st.vx;
            sl.ay = X.y - st.vy;
        }
        double bx, by;
        rc = gdt_tile_search_f64<1, CERT, GEN>(S, L, sl, npred, 0, false, bk, bx, by, st.tbl,
                                          (unsigned)tot, ph, &io);
    }
    int res = STEP_RUN;
    if (CERT && !gdt_tile_x_range(S, io, L.orig[st.iv])) {
        res = STEP_DEFER;
    } else if (tot > 64) {
        if (lane == 0) {
            int r = STEP_RUN;
            while (r == STEP_RUN) r = gdt_tile_step_f64<1, CERT, GEN>(S, L, io, st, npred);
            res = r;
            count = st.count;
        }
    } else {
        const unsigned long long mv = __ballot(kg == st.iv);
        const int hv = __ffsll((long long)mv) - 1;
        int nn = __shfl(bk, hv, 64), nrc = __shfl(rc, hv, 64);
        if (nrc != STEP_RUN) {
            // not certified over the block: lane 0 runs the full search
            if (lane == 0) {
                double bx, by;
                nrc = gdt_tile_search_f64<1, CERT, GEN>(S, L, st, npred, 0, true, nn, bx, by,
                                                   nullptr, 0, GDT_SCAN0, &io);
            }
            nrc = __shfl(nrc, 0, 64);
            nn = __shfl(nn, 0, 64);
        }
        if (nrc != STEP_RUN) {
            res = STEP_DEFER;
        } else {
            if (lane == 0) st.row[0] = L.orig[nn];
            count = 1;
            for (int cur = nn;;) {
                const unsigned long long m = __ballot(kg == cur && rc == STEP_RUN);
                int nx;
                if (m) {
                    nx = __shfl(bk, __ffsll((long long)m) - 1, 64);
                } else {
                    // no lane certified cur's successor: lane 0 runs the
                    // full search from cur (extension included)
                    int r = STEP_DEFER, b = -1;
                    if (lane == 0) {
                        GdtTileLane<double> sl = st;
                        const gdt_d2 X = L.X64[cur];
                        sl.ak = cur;
                        sl.ax = X.x - st.vx;
                        sl.ay = X.y - st.vy;
                        double bx, by;
                        r = gdt_tile_search_f64<1, CERT, GEN>(S, L, sl, npred, 0, true, b, bx, by,
                                                         nullptr, 0, GDT_SCAN0, &io);
                    }
                    if (__shfl(r, 0, 64) != STEP_RUN) {
                        res = STEP_DEFER;
                        break;
                    }
                    nx = __shfl(b, 0, 64);
                }
                if (nx == nn) {
                    res = STEP_DONE;
                    break;
                }
                if (lane == 0 && count < io.stride) st.row[count] = L.orig[nx];
                if (++count > GDT_HARD_CAP) {
                    res = STEP_NOCLOSE;
                    break;
                }
                cur = nx;
            }
        }
    }
    if (CERT && res == STEP_DEFER) tied = __any(bk == GDT_TIE);
    return res;
}

// Points of a tile left by the hull routine that go straight to wavefronts (at most).
#define GDT_HULL_WAVES 16
// Records of points with open triangles a block keeps (32x32-cell tiles of random
// points have about 200 of one point to a cell, 280 of 1.2, and in the larger
// windows 480 of 1.44 and 700 of 2).
#ifdef GDT_WIN_DENSE
#define GDT_HULL_RECS 640
#else
#define GDT_HULL_RECS 256
#endif
// Records a wave closes together.
#define GDT_HULL_TAKE 32

// One block per tile, one point per lane: the hull routine (gdt_hull.h) over
// all of the tile's points -- or, with `flags`, the flagged ones, as
// k_one_ring_tile.  Waves take 64 points at a time; those with open triangles
// (a fifth of random points) are recorded in LDS, so that full waves close them,
// where every wave would wait for its few.  The points left to the steps (under
// 0.1 % of random points) take them, or when they are few a wavefront's star
// search each.
// (Overfull pools that left points to the steps cost more at other cell sizes: 2^20
// points of 1.2 to a cell 648 us per call, now 540, of 1.44 680 and 508, of 0.64 990
// and 757.)
// Bound by the vector ALU and by the imbalance of its parts (a 1M-point tile:
// 9 us for staging, 65 for the lists, 39 for the open triangles, and 40 more in
// the third of the tiles with a point left; FP64 adds and multiplies are half of
// the instructions), not by memory (0.14 GB, 20 us).  Ring kernel of 1M / 3.9M
// uniform points 342 / 1,155 us (the steps: 496 / 1,890 at 4M), of a 1M
// near-lattice 228 (339).  Blocks of 512, two
// to a compute unit: 1,024 threads took 477 us at 1M, 256 threads on 16x16
// tiles 445, 320 threads 622; a cap of 96 registers for five waves spilled
// (421).  Closing by each wave for its own lanes took 375 us, by single lanes
// after a barrier 493, in block-wide rounds 460; without the drain before the
// barrier 384.
template <bool GEN>
__global__ __launch_bounds__(1024) void k_one_ring_hull(const GdtSet* __restrict__ sets,
                                                        const GdtChunk* __restrict__ tiles,
                                                        const int* __restrict__ flags,
                                                        const int* __restrict__ halt, GdtRingIO io,
                                                        int* __restrict__ counts,
                                                        int* __restrict__ status,
                                                        unsigned long long* __restrict__ counters,
                                                        int* __restrict__ defer)
{
    __shared__ uint32_t s_cs[GDT_WIN_CELLS + 1];
    __shared__ gdt_d2 s_X64[GDT_WIN_MAXPTS + 1];
    __shared__ int s_orig[GDT_WIN_MAXPTS];
    __shared__ uint32_t s_wsum[16];
    __shared__ int s_next, s_next2, s_rn, s_rt;
    __shared__ int s_dlist[GDT_TILE_DEFER];
    __shared__ uint32_t s_dn;
    __shared__ unsigned long long s_fmask[GDT_WIN_MAXPTS / 64], s_smask[GDT_WIN_MAXPTS / 64];
    __shared__ uint32_t s_fpre[GDT_WIN_MAXPTS / 64 + 1], s_spre[GDT_WIN_MAXPTS / 64 + 1];
    __shared__ uint32_t s_rec[GDT_HULL_REC * GDT_HULL_RECS];
    // [2 GDT_HULL_GROUPS * waves] the waves' queues, [GDT_HULL_WORDS * blockDim + 1] lists
    extern __shared__ uint32_t s_dyn[];

    const GdtChunk ch = tiles[blockIdx.x];
    const GdtSet S = sets[ch.set];
    const GdtTileWin w = gdt_tile_window(S, ch.start);
    GdtTileLds L;
    L.cs = s_cs; L.gstart = nullptr; L.X64 = s_X64; L.X32 = nullptr; L.orig = s_orig;
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63;
    const int k0 = S.c0 + ch.start * GDT_TILE_CELLS;
    const int T0 = (int)io.cstart[k0], T1 = (int)io.cstart[k0 + GDT_TILE_CELLS];
    const int npt = T1 - T0;
    if (flags && halt && *halt) return;
    TileFlags tf = {s_fmask, s_fpre, 0};
    int Q0 = T0, Q1 = T1;
    if (flags && npt <= GDT_WIN_MAXPTS) {
        Q0 = 0;
        Q1 = tile_gather_flags(flags, io.perm, T0, npt, s_fmask, s_fpre, tf);
        if (tid == 0 && Q1 > 0) atomicAdd(&status[ST_NFLAGGED], Q1);
    }
    auto item = [&](int q) { return tf.nw ? tile_flagged_slot(tf, T0, q) : q; };
    if (Q0 >= Q1) return;    // block-uniform: nothing to do in this tile

    const bool fits = npt <= GDT_WIN_MAXPTS && gdt_stage_window<false, GEN>(S, w, io, L, s_wsum);
    if (!fits) {
        unsigned nf = 0;
        for (int q = Q0 + tid; q < Q1; q += nt) {
            const int j = item(q);
            if (flags && !tf.nw) {      // (more points than a window holds: no mask)
                if (flags[io.perm[j]] < 0) continue;
                ++nf;
            }
            const uint32_t pos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u);
            defer[pos] = j;
        }
        if (nf) atomicAdd(&status[ST_NFLAGGED], (int)nf);
        return;
    }
    if (tid == 0) {
        s_next = s_next2 = s_rn = s_rt = 0;
        s_dn = 0u;
    }
    const int nsw = (npt + 63) >> 6;
    for (int t = tid; t < nsw; t += nt) s_smask[t] = 0ull;
    for (int t = tid; t < GDT_HULL_RECS; t += nt) s_rec[GDT_HULL_REC * t + 1] = 0u;
    __syncthreads();
    uint32_t* const wq = s_dyn + 2 * GDT_HULL_GROUPS * (tid >> 6);
    uint32_t* const wave_words =
        s_dyn + 2 * GDT_HULL_GROUPS * (nt >> 6) + GDT_HULL_WORDS * (tid - lane);
    uint32_t* const words = wave_words + GDT_HULL_WORDS * lane;
    unsigned npred = 0, nsum = 0;
    int mx = 0, er = 0;
    // entry iv's row from the list in the lane's words
    auto emit = [&](int iv, int n) {
        const int i = L.orig[iv];
        int* row = io.nbrs + (size_t)i * (size_t)io.stride;
        for (int m = 0; m < n && m < io.stride; ++m) row[m] = L.orig[gdt_hull_entry(words, m)];
        counts[i] = n;
        mx = max(mx, n);
        nsum += (unsigned)n;
    };
    auto lane_init = [&](GdtTileLane<double>& st, int j) {
        if constexpr (GEN) gdt_tile_lane_init_gen(w, L, j, io, S, st);
        else gdt_tile_lane_init<double>(w, L, j, io, S, st);
    };
    // slot j's point is left to the steps
    auto leave = [&](int j) { atomicOr(&s_smask[(j - T0) >> 6], 1ull << ((j - T0) & 63)); };
    // the wave's points (`mine`: this lane has one) closed, and their rows
    auto close = [&](bool mine, GdtHull& h, int iv, int c0) {
        gdt_hull_close_wave<GEN>(S, L, iv, c0, wave_words, wq, h, npred);
        if (!mine) return;
        if (!h.bad) {
            emit(iv, h.n);
        } else {
            // its slot: the cell's first slot plus the rank in the cell
            leave((int)io.cstart[gdt_tile_key(S, w, c0)] + iv - (int)L.cs[c0]);
        }
    };
    // (cells of more than two points: what a 3x3 block leaves open is a third of the
    // points, whose steps, all at once, take less than their closing: 2^20 points of 2.25
    // to a cell 700 us per call, 787 closed; of 1.7 to a cell 622 closed, 780 by steps)
    const bool full = npt > 2 * GDT_TILE_CELLS;
    for (;;) {
        int c = 0;
        if (lane == 0) c = atomicAdd(&s_next, 64);
        const int q = Q0 + __builtin_amdgcn_readfirstlane(c) + lane;
        if (q - lane >= Q1) break;      // (wave-uniform)
        GdtHull h = {0, 0, 0u, true, 0.};
        int iv = 0, c0 = 0;
        bool mine = false;
        if (q < Q1) {
            const int j = item(q);
            GdtTileLane<double> st;
            lane_init(st, j);
            gdt_hull_build<GEN>(S, L, st, words, h, npred);
            if (h.bad || (full && h.open != 0)) {
                leave(j);
                h.open = 0;
            } else if (h.open == 0) {
                emit(st.iv, h.n);
            } else {
                const int r = atomicAdd(&s_rn, 1);
                mine = r >= GDT_HULL_RECS;
                iv = st.iv;
                c0 = st.c0;
                if (!mine) {
                    gdt_hull_save(h, iv, c0, words, s_rec + GDT_HULL_REC * r);
                    h.open = 0;
                }
            }
        }
        // (no room among the records: closed by this wave; which points these are
        // is up to the waves' order, but not what a row is)
        if (__any(mine)) close(mine, h, iv, c0);
    }
    // Records are closed by the waves that have no chunk left, while others
    // still run theirs, and after a barrier the last ones.
    auto drain = [&](int most) {
        for (;;) {
            int t = 0, take = 0;
            if (lane == 0) {
                t = __hip_atomic_load(&s_rt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                for (;;) {
                    const int n = min(__hip_atomic_load(&s_rn, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP),
                                      GDT_HULL_RECS);
                    take = min(most, n - t);
                    if (take <= 0) break;
                    const int seen = atomicCAS(&s_rt, t, t + take);
                    if (seen == t) break;
                    t = seen;
                }
            }
            t = __builtin_amdgcn_readfirstlane(t);
            take = __builtin_amdgcn_readfirstlane(take);
            if (take <= 0) break;
            GdtHull h = {0, 0, 0u, true, 0.};
            int iv = 0, c0 = 0;
            if (lane < take) {
                const uint32_t* rec = s_rec + GDT_HULL_REC * (t + lane);
                // (its wave reserved it just before it writes it)
                while (__hip_atomic_load(rec + 1, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) == 0u)
                    __builtin_amdgcn_s_sleep(1);
                gdt_hull_load(L, rec, h, iv, c0, words);
            }
            close(lane < take, h, iv, c0);
        }
    };
    // (a repair's few are shared out by all of the waves, most of which had no
    // chunk)
    if (flags) __syncthreads();
    for (int last = flags ? 1 : 0; last < 2; ++last) {
        const int nw = nt >> 6;
        drain(flags ? min(GDT_HULL_TAKE, max(1, (min(s_rn, GDT_HULL_RECS) + nw - 1) / nw)) : GDT_HULL_TAKE);
        __syncthreads();
    }
    // The points left to the steps, as in k_one_ring_tile.  Few of them take a
    // wavefront each, as the star kernel's points: one search's chain for the
    // ring, and one more where a circle leaves the lanes' block, not a chain of
    // searches (a tile in three has such a point, and ends with it).
    TileFlags sf = {s_smask, s_spre, nsw};
    const int nslow = tile_mask_prefix(sf, s_spre);
    if (nslow > 0 && nslow <= GDT_HULL_WAVES) {
        for (int t = tid >> 6; t < nslow; t += nt >> 6) {       // (wave-uniform)
            const int j = tile_flagged_slot(sf, T0, t);
            GdtTileLane<double> st;
            st.tbl = words;
            lane_init(st, j);
            int count = 0;
            bool tied = false;
            const int res = star_ring<false, GEN>(S, L, io, st, npred, count, tied);
            if (lane == 0) {
                if (res == STEP_DEFER) {
                    s_dlist[atomicAdd(&s_dn, 1u)] = j;
                } else {
                    counts[L.orig[st.iv]] = count;
                    mx = max(mx, count);
                    nsum += (unsigned)count;
                    if (res == STEP_NOCLOSE) er |= ERR_NOCLOSE;
                }
            }
        }
    } else if (nslow > 0) {
        int q = tid;
        bool have = q < nslow;
        int j = 0;
        GdtTileLane<double> st;
        st.tbl = words;
        if (have) {
            j = tile_flagged_slot(sf, T0, q);
            lane_init(st, j);
        }
        // (clumps in a general box are handed on: their steps are long chains, and
        // its lists go one lane each: 262,144 points, half of them in 200 clumps,
        // 6.6 ms per call with the steps, 5.0 without)
        auto clumped = [&]() {
            int n = 0;
            for (int r = -1; r <= 1; ++r) {
                const uint32_t* row = L.cs + st.c0 + r * GDT_WIN;
                n += (int)(row[2] - row[-1]);
            }
            return n > GDT_HULL_SLOTS;
        };
        while (__ballot(have) != 0) {
            if (have) {
                const bool hand_on = GEN && clumped();
                const int rc = hand_on ? STEP_DEFER
                                       : gdt_tile_step_f64<1, false, GEN>(S, L, io, st, npred);
                if (rc != STEP_RUN) {
                    if (rc == STEP_DEFER) {
                        const uint32_t dpos = hand_on ? GDT_TILE_DEFER : atomicAdd(&s_dn, 1u);
                        if (dpos < GDT_TILE_DEFER) {
                            s_dlist[dpos] = j;
                        } else {
                            const uint32_t pos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u);
                            defer[pos] = j;
                        }
                    } else {
                        counts[L.orig[st.iv]] = st.count;
                        mx = max(mx, st.count);
                        nsum += (unsigned)st.count;
                        if (rc == STEP_NOCLOSE) er |= ERR_NOCLOSE;
                    }
                    q = nt + atomicAdd(&s_next2, 1);
                    have = q < nslow;
                    if (have) {
                        j = tile_flagged_slot(sf, T0, q);
                        lane_init(st, j);
                    }
                }
            }
        }
    }
    __syncthreads();
    tile_finish_deferred<GEN>(S, io, s_dlist, min((int)s_dn, GDT_TILE_DEFER), counts, status, defer,
                              npred, nsum, mx, er);
    ring_block_totals(mx, er, npred, 0u, nsum, status, counters);
}

// One wavefront per point (small grids; FP64 predicates): lane g takes entry g
// of the cell block around the point's cell (7x7 cells, or 5x5 when the 7x7
// block holds more than 64 entries), in the order a step scans it, and runs
// the step's search (gdt_tile_search_f64) over that block with that
// candidate as the current neighbour -- every candidate's successor at once;
// the lane holding the point itself runs the nearest-neighbour search.  The
// ring is then the walk nearest -> successor -> ... read from the lanes: the
// sequential walk, each step's result taken from the lane that ran the same
// search on the same state.  Where the walk reaches a candidate whose search
// the lanes did not certify (its circle leaves the block: those lanes do not
// extend) or one outside the block, lane 0 runs that one search in full; a
// block of more than 64 entries runs the sequential steps in lane 0.  Blocks
// (tile, y) share a tile's points: wave w of block y takes the points
// T0 + y nw + w + m gridDim.y nw.  Deferred points go to `defer` (handled by
// k_one_ring_deferred in the next launch); the exact mode's, which may be all of a
// lattice, a block's together (an atomic for each took 160 of 195 us where all of
// 16,384 points were handed on).
template <bool CERT, bool GEN = false>
__global__ __launch_bounds__(CERT ? GDT_XTILE_BLOCK : 1024) void k_one_ring_star(const GdtSet* __restrict__ sets,
                                                        const GdtChunk* __restrict__ tiles,
                                                        GdtRingIO io, int* __restrict__ counts,
                                                        int* __restrict__ status,
                                                        unsigned long long* __restrict__ counters,
                                                        int* __restrict__ defer)
{
    __shared__ uint32_t s_cs[GDT_WIN_CELLS + 1];
    __shared__ gdt_d2 s_X64[GDT_WIN_MAXPTS + 1];
    __shared__ gdt_f2 s_X32[1];
    __shared__ int s_orig[GDT_WIN_MAXPTS];
    __shared__ uint32_t s_wsum[16];
    __shared__ int s_hand[CERT ? STAR_HAND : 1];
    __shared__ uint32_t s_hn, s_hpos;
    extern __shared__ uint32_t s_tbl[];     // [STAR_TBL * blockDim + 1] the lanes' row tables

    const GdtChunk ch = tiles[blockIdx.x];
    const GdtSet S = sets[ch.set];
    const GdtTileWin w = gdt_tile_window(S, ch.start);
    GdtTileLds L;
    L.cs = s_cs; L.gstart = nullptr; L.X64 = s_X64; L.X32 = s_X32; L.orig = s_orig;
    const int tid = threadIdx.x, lane = tid & 63, nw = (int)blockDim.x >> 6;
    const int k0 = S.c0 + ch.start * GDT_TILE_CELLS;
    const int T0 = (int)io.cstart[k0], T1 = (int)io.cstart[k0 + GDT_TILE_CELLS];
    const int qstep = (int)gridDim.y * nw;
    const int qb = T0 + (int)blockIdx.y * nw;
    if (qb >= T1) return;    // block-uniform: no point for this block

    const bool fits = gdt_stage_window<false, GEN>(S, w, io, L, s_wsum);
    if (!fits) {
        if (lane == 0)
            for (int q = qb + (tid >> 6); q < T1; q += qstep) {
                const uint32_t pos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u);
                defer[pos] = q;
            }
        return;
    }
    if constexpr (CERT) {
        if (tid == 0) s_hn = 0u;
        __syncthreads();
    }
    auto hand_on = [&](int q) {
        const uint32_t h = CERT ? atomicAdd(&s_hn, 1u) : STAR_HAND;
        if (h < STAR_HAND) s_hand[h] = q;
        else defer[atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), 1u)] = q;
    };
    unsigned npred = 0, nsum = 0;
    int mx = 0, er = 0;
    for (int q = qb + (tid >> 6); q < T1; q += qstep) {     // wave-uniform
        GdtTileLane<double> st;
        st.tbl = s_tbl + STAR_TBL * tid;
        if constexpr (GEN) gdt_tile_lane_init_gen(w, L, q, io, S, st);
        else gdt_tile_lane_init<double>(w, L, q, io, S, st);
        int count = 0;
        bool tied = false;
        const int res = star_ring<CERT, GEN>(S, L, io, st, npred, count, tied);
        if (CERT && tied) {
            // (ties come by the lattice: the wave's other points are handed on unseen)
            for (int p = q + lane * qstep; p < T1; p += 64 * qstep) hand_on(p);
            break;
        }
        if (lane == 0) {
            if (res == STEP_DEFER) {
                hand_on(q);
            } else {
                counts[L.orig[st.iv]] = count;
                mx = max(mx, count);
                nsum += (unsigned)count;
                if (res == STEP_NOCLOSE) er |= ERR_NOCLOSE;
            }
        }
    }
    if constexpr (CERT) {
        __syncthreads();
        const int nh = min((int)s_hn, STAR_HAND);
        if (nh > 0) {       // (block-uniform)
            if (tid == 0)
                s_hpos = atomicAdd(reinterpret_cast<unsigned int*>(&status[ST_NDEFER]), (unsigned)nh);
            __syncthreads();
            for (int t = tid; t < nh; t += (int)blockDim.x) defer[s_hpos + t] = s_hand[t];
        }
    }
    ring_block_totals(mx, er, npred, 0u, nsum, status, counters);
}

hipError_t gdt_launch_one_ring_tile(int precision, const GdtSet* d_sets, int nsets,
                                    const GdtChunk* tiles, int ntiles, int block, int lanes,
                                    bool general,
                                    const int* flags, const int* halt,
                                    const GdtRingIO& io, int* counts, int* status,
                                    unsigned long long* counters, int* defer, int rest,
                                    hipEvent_t after_tile, hipStream_t s)
{
    if (ntiles <= 0) return hipSuccess;
    if (block > 1024) block = 1024;
    if (precision == GDT_EXACT && block > GDT_XTILE_BLOCK) block = GDT_XTILE_BLOCK;
    if (general && precision != 64) return hipErrorInvalidValue;
    // One lane per point, FP64 and FP32-filtered alike: the hull kernel, whose
    // FP64 rows are the filtered path's too.  (Ring kernel of 1M uniform points
    // 342 us; the search steps took 496 in FP64 and 544 filtered.)
#ifdef GDT_WIN_DENSE
    // (windows of 4,096 points take a compute unit's LDS: one block of them)
    block = precision == GDT_EXACT ? GDT_XTILE_BLOCK : 1024;
    const bool hull = precision != GDT_EXACT;
#else
    const bool hull = precision != GDT_EXACT && lanes == 1;
#endif
    const size_t tbl = (5 * (size_t)block + 1) * sizeof(uint32_t);
    if (hull) {
        const size_t words = (2 * GDT_HULL_GROUPS * (size_t)(block >> 6) +
                              GDT_HULL_WORDS * (size_t)block + 1) * sizeof(uint32_t);
        auto* k = general ? k_one_ring_hull<true> : k_one_ring_hull<false>;
        hipLaunchKernelGGL(k, dim3(ntiles), dim3(block), words, s, d_sets, tiles, flags, halt, io,
                           counts, status, counters, defer);
    } else {
        auto* k = k_one_ring_tile<GDT_EXACT, 1>;
#ifndef GDT_WIN_DENSE
        if (precision == GDT_EXACT && lanes > 1)
            k = k_one_ring_tile<GDT_EXACT, 2>;
        else if (precision == 32)
            k = k_one_ring_tile<32, 2>;
        else if (precision == 64)
            // (four lanes per point: in a rectangle only; elsewhere two)
            k = general ? k_one_ring_tile<64, 2, true>
                        : (lanes == 4 ? k_one_ring_tile<64, 4> : k_one_ring_tile<64, 2>);
#endif
        hipLaunchKernelGGL(k, dim3(ntiles), dim3(block), tbl, s, d_sets, tiles, flags, halt, io,
                           counts, status, counters, defer);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (after_tile && (e = hipEventRecord(after_tile, s)) != hipSuccess) return e;
    return gdt_launch_deferred(precision, d_sets, nsets, io, counts, status, counters,
                               defer, rest, s);
}

#ifndef GDT_WIN_DENSE
hipError_t gdt_launch_one_ring_star(int precision, const GdtSet* d_sets, int nsets,
                                    const GdtChunk* tiles,
                                    int ntiles, int nsplit, int block, bool general,
                                    const GdtRingIO& io, int* counts, int* status,
                                    unsigned long long* counters, int* defer, int rest,
                                    hipEvent_t after_tile, hipStream_t s)
{
    if (ntiles <= 0) return hipSuccess;
    if (block < 64 || block > 1024 || (block & 63) || nsplit < 1 || nsplit > 65535)
        return hipErrorInvalidValue;
    const size_t tbl = (STAR_TBL * (size_t)block + 1) * sizeof(uint32_t);
    if (precision == GDT_EXACT && block > GDT_XTILE_BLOCK) return hipErrorInvalidValue;
    if (general && precision != 64) return hipErrorInvalidValue;
    if (general)
        hipLaunchKernelGGL((k_one_ring_star<false, true>), dim3(ntiles, nsplit), dim3(block), tbl,
                           s, d_sets, tiles, io, counts, status, counters, defer);
    else if (precision == GDT_EXACT)
        hipLaunchKernelGGL(k_one_ring_star<true>, dim3(ntiles, nsplit), dim3(block), tbl, s, d_sets,
                           tiles, io, counts, status, counters, defer);
    else
        hipLaunchKernelGGL(k_one_ring_star<false>, dim3(ntiles, nsplit), dim3(block), tbl, s,
                           d_sets, tiles, io, counts, status, counters, defer);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (after_tile && (e = hipEventRecord(after_tile, s)) != hipSuccess) return e;
    return gdt_launch_deferred(precision == GDT_EXACT ? GDT_EXACT : 64, d_sets, nsets, io, counts,
                               status, counters, defer, rest, s);
}
#endif

}  // namespace GDT_TS_NS
