// onering.hip -- per-point Delaunay one-ring kernels (FP64 and FP32-filtered)
// and the wavefront kernel of the points the LDS tile kernel (tile.hip) defers.
//
// One lane per point.  Lanes of a block take consecutive cell-ordered slots,
// so a wavefront covers a compact patch of cells (8x8-cell tiles by default)
// and the candidate offsets it reads come from the same few cache lines.
// Replaces gpu_voronoi_calc_global_kernel + gpu_get_neighbors_global_kernel
// (DelaunayGPU.cu:649-675, 981-1006) and their masked repair variants
// (DelaunayGPU.cu:611-640, 945-975), which instead launch every point and
// mask most of them out.
#include "gdt_exact_wave.h"
#include "gdt_kernels.h"
#include "gdt_wavedev.h"

#include <type_traits>

template <int PREC>
__device__ inline GdtRingResult ring_of(const GdtSet& S, int j, const GdtRingIO& io)
{
    if constexpr (PREC == GDT_EXACT) return gdt_one_ring_exact(S, j, io);
    else return PREC == 32 ? gdt_one_ring_f32(S, j, io) : gdt_one_ring_f64(S, j, io);
}

// The totals of a wave's results (every lane of the wave calls it).
__device__ inline void ring_wave_totals(bool active, const GdtRingResult& r, int* __restrict__ status,
                                        unsigned long long* __restrict__ counters)
{
    const int mx = wave_max_i32(r.count);
    const int er = wave_or_i32(r.err);
    const unsigned np = wave_sum_u32(r.npred);
    const unsigned nf = wave_sum_u32(r.nfb);
    const unsigned ns = wave_sum_u32(active ? (unsigned)r.count : 0u);
    if ((threadIdx.x & 63) == 0) {
        if (mx > 0) atomicMax(&status[ST_REQUIRED], mx);
        if (er) atomicOr(&status[ST_ERRFLAGS], er);
        if (np) atomicAdd(&counters[CT_PRED], (unsigned long long)np);
        if (nf) atomicAdd(&counters[CT_FALLBACK], (unsigned long long)nf);
        if (ns) atomicAdd(&counters[CT_NBRSUM], (unsigned long long)ns);
    }
}

// A point whose search the grid's search radius cannot certify (boxes of a
// few cells) is appended to `defer` (when given) for the wavefront kernel,
// whose searches may stop at the cell box of their circle; its row is then
// rewritten there.
template <int PREC>
__device__ inline void one_ring_lane(bool active, const GdtSet& S, int j, const GdtRingIO& io,
                                     int* __restrict__ counts, int* __restrict__ status,
                                     unsigned long long* __restrict__ counters,
                                     int* __restrict__ defer)
{
    GdtRingResult r = {0, 0, 0u, 0u};
    if (active) {
        r = ring_of<PREC>(S, j, io);
        if (defer && (r.err & ERR_SEARCH)) {
            defer[atomicAdd(reinterpret_cast<unsigned*>(status + ST_NDEFER), 1u)] = j;
            r.count = 0;
            r.err = 0;
        } else {
            counts[io.perm[j]] = r.count;
        }
    }
    ring_wave_totals(active, r, status, counters);
}

// All points: block b handles chunk b (one set, blockDim consecutive slots).
template <int PREC>
__global__ __launch_bounds__(1024) void k_one_ring(const GdtSet* __restrict__ sets,
                                                   const GdtChunk* __restrict__ chunks,
                                                   GdtRingIO io, int* __restrict__ counts,
                                                   int* __restrict__ status,
                                                   unsigned long long* __restrict__ counters,
                                                   int* __restrict__ defer)
{
    const GdtChunk ch = chunks[blockIdx.x];
    const GdtSet S = sets[ch.set];
    const int li = ch.start + (int)threadIdx.x;
    const bool active = li < S.n;
    one_ring_lane<PREC>(active, S, S.p0 + li, io, counts, status, counters, defer);
}

// Entries [first, len) of a slot list, one lane each over the grid, set found
// per lane (ONE: a single set, which then stays in scalar registers).
template <int PREC, bool ONE = false>
__device__ inline void one_ring_lanes(const GdtSet* __restrict__ sets, int nsets,
                                      const int* __restrict__ worklist, int first, int len,
                                      const GdtRingIO& io, int* __restrict__ counts,
                                      int* __restrict__ status,
                                      unsigned long long* __restrict__ counters,
                                      int* __restrict__ defer)
{
    const int stride = gridDim.x * blockDim.x;
    // uniform trip count per wave so the reductions see every lane
    const int wave_first = first + (int)(blockIdx.x * blockDim.x + (threadIdx.x & ~63u));
    for (int base = wave_first; base < len; base += stride) {
        const int t = base + (int)(threadIdx.x & 63);
        const bool active = t < len;
        const int j = active ? worklist[t] : 0;
        const GdtSet S = sets[ONE || !active ? 0 : gdt_set_of(sets, nsets, j)];
        one_ring_lane<PREC>(active, S, j, io, counts, status, counters, defer);
    }
}

// Entries from `first` of a worklist of slots (count in device memory), one lane each.
// ONE: a single set (FP64: 68 registers and seven waves to a SIMD, 94 and five
// with a set per lane).  THREADS: the largest block; at 256 the exact routine
// keeps its registers, at 1,024 it spills some for twice the waves
// (GDT_XLIST_SHORT).
template <int PREC, bool ONE, int THREADS = 1024>
__global__ __launch_bounds__(THREADS) void k_one_ring_list(const GdtSet* __restrict__ sets, int nsets,
                                                        const int* __restrict__ worklist,
                                                        const uint32_t* __restrict__ worklen,
                                                        GdtRingIO io, int* __restrict__ counts,
                                                        int* __restrict__ status,
                                                        unsigned long long* __restrict__ counters,
                                                        int* __restrict__ defer, int first)
{
    one_ring_lanes<PREC, ONE>(sets, nsets, worklist, first, (int)*worklen, io, counts, status, counters,
                         defer);
}

// Deferred points (count in device memory): the first `cap` one wavefront
// each, grid-stride over the waves (FP64 in both precision paths; exact
// decisions in the exact mode), and, where `rest` says so, any beyond (dense
// clusters) one lane each, and again by the wavefront where the lane's search does
// not certify a circle; GDT_LIST_LATER: none of a longer list.
template <int PREC>
__global__ __launch_bounds__(256) void k_one_ring_deferred(const GdtSet* __restrict__ sets,
                                                           int nsets,
                                                           const int* __restrict__ worklist,
                                                           const uint32_t* __restrict__ worklen,
                                                           int cap, GdtRingIO io,
                                                           int* __restrict__ counts,
                                                           int* __restrict__ status,
                                                           unsigned long long* __restrict__ counters,
                                                           int rest)
{
    const int lane = (int)(threadIdx.x & 63);
    const int wid = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int nw = (int)((gridDim.x * blockDim.x) >> 6);
    const int all = (int)*worklen;
    const int len = rest == GDT_LIST_LATER && all > cap ? 0 : min(all, cap);
    GdtWaveDev w;
    w.lane = lane;
    unsigned npred = 0, nsum = 0;
    int mx = 0, er = 0;
    for (int t = wid; t < len; t += nw) {
        const int j = worklist[t];
        const GdtSet S = sets[gdt_set_of(sets, nsets, j)];
        GdtRingResult r;
        if constexpr (PREC == GDT_EXACT)
            r = gdt_wave_ring_exact(S, j, io, w, lane == 0);
        else
            r = gdt_wave_ring(S, j, io, w, lane == 0);
        npred += r.npred;
        er |= r.err;
        if (lane == 0) {
            counts[io.perm[j]] = r.count;
            mx = max(mx, r.count);
            nsum += (unsigned)r.count;
        }
    }
    if (wid < len) {        // (wave-uniform)
        mx = wave_max_i32(mx);
        er = wave_or_i32(er);
        npred = wave_sum_u32(npred);
        nsum = wave_sum_u32(nsum);
        if (lane == 0) {
            if (mx > 0) atomicMax(&status[ST_REQUIRED], mx);
            if (er) atomicOr(&status[ST_ERRFLAGS], er);
            if (npred) atomicAdd(&counters[CT_PRED], (unsigned long long)npred);
            if (nsum) atomicAdd(&counters[CT_NBRSUM], (unsigned long long)nsum);
        }
    }
    if constexpr (PREC != GDT_EXACT) {
        if (rest != GDT_REST_HERE) return;
        for (int base = len + 64 * wid; base < all; base += 64 * nw) {      // (wave-uniform)
            const bool active = base + lane < all;
            const int j = active ? worklist[base + lane] : 0;
            GdtRingResult r = {0, 0, 0u, 0u};
            if (active) r = ring_of<PREC>(sets[gdt_set_of(sets, nsets, j)], j, io);
            for (unsigned long long m = __ballot((r.err & ERR_SEARCH) != 0); m; m &= m - 1ull) {
                const int from = __ffsll((long long)m) - 1, jw = __shfl(j, from, 64);
                const GdtSet S = sets[gdt_set_of(sets, nsets, jw)];
                const GdtRingResult g = gdt_wave_ring(S, jw, io, w, lane == 0);
                r.npred += g.npred;
                if (lane == from) {
                    r.count = g.count;
                    r.err = g.err;
                }
            }
            if (active) counts[io.perm[j]] = r.count;
            ring_wave_totals(active, r, status, counters);
        }
    }
}

hipError_t gdt_launch_deferred(int precision, const GdtSet* d_sets, int nsets,
                               const GdtRingIO& io, int* counts, int* status,
                               unsigned long long* counters, int* defer, int rest, hipStream_t s)
{
    if (precision == GDT_EXACT && rest != GDT_LIST_LATER) return hipErrorInvalidValue;
    const int cap = gdt_wave_cap(precision);
    // (the count is read on the device)
    const uint32_t* ndefer = reinterpret_cast<const uint32_t*>(status + ST_NDEFER);
    if (precision == 32)
        hipLaunchKernelGGL(k_one_ring_deferred<32>, dim3(GDT_WAVE_BLOCKS), dim3(256), 0, s, d_sets,
                           nsets, defer, ndefer, cap, io, counts, status, counters, rest);
    else if (precision == GDT_EXACT)
        hipLaunchKernelGGL(k_one_ring_deferred<GDT_EXACT>, dim3(GDT_WAVE_BLOCKS), dim3(256), 0, s,
                           d_sets, nsets, defer, ndefer, cap, io, counts, status, counters,
                           rest);
    else
        hipLaunchKernelGGL(k_one_ring_deferred<64>, dim3(GDT_WAVE_BLOCKS), dim3(256), 0, s, d_sets,
                           nsets, defer, ndefer, cap, io, counts, status, counters, rest);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || rest <= 0) return e;
    return gdt_launch_one_ring(precision, d_sets, nsets, nullptr, 0, 256, defer, ndefer, cap, rest,
                               io, counts, status, counters, nullptr, s);
}

hipError_t gdt_launch_deferred_rest(int precision, const GdtSet* d_sets, int nsets, int first,
                                    int len, const GdtRingIO& io, int* counts, int* status,
                                    unsigned long long* counters, const int* defer, hipStream_t s)
{
    return gdt_launch_one_ring(precision, d_sets, nsets, nullptr, 0, 256, defer,
                               reinterpret_cast<const uint32_t*>(status + ST_NDEFER), first, len, io,
                               counts, status, counters, nullptr, s);
}

hipError_t gdt_launch_one_ring(int precision, const GdtSet* d_sets, int nsets,
                               const GdtChunk* chunks, int nch, int block, const int* worklist,
                               const uint32_t* worklen, int first, int max_work,
                               const GdtRingIO& io, int* counts, int* status,
                               unsigned long long* counters, int* defer, hipStream_t s)
{
    if (!worklist) {
        if (nch <= 0) return hipSuccess;
        if (precision == 32)
            hipLaunchKernelGGL(k_one_ring<32>, dim3(nch), dim3(block), 0, s, d_sets, chunks, io,
                               counts, status, counters, defer);
        else if (precision == GDT_EXACT)
            hipLaunchKernelGGL(k_one_ring<GDT_EXACT>, dim3(nch), dim3(block), 0, s, d_sets,
                               chunks, io, counts, status, counters, defer);
        else
            hipLaunchKernelGGL(k_one_ring<64>, dim3(nch), dim3(block), 0, s, d_sets, chunks, io,
                               counts, status, counters, defer);
        return hipGetLastError();
    }
    max_work -= first;
    if (max_work <= 0) return hipSuccess;
    int grid = (max_work + block - 1) / block;
    if (grid > 4096) grid = 4096;
    const bool one = nsets == 1;
    auto* k = one ? k_one_ring_list<64, true> : k_one_ring_list<64, false>;
    if (precision == 32)
        k = one ? k_one_ring_list<32, true> : k_one_ring_list<32, false>;
    else if (precision == GDT_EXACT && block <= 256 && max_work <= GDT_XLIST_SHORT)
        k = one ? k_one_ring_list<GDT_EXACT, true, 256> : k_one_ring_list<GDT_EXACT, false, 256>;
    else if (precision == GDT_EXACT)
        k = one ? k_one_ring_list<GDT_EXACT, true> : k_one_ring_list<GDT_EXACT, false>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(block), 0, s, d_sets, nsets, worklist, worklen, io, counts,
                       status, counters, defer, first);
    return hipGetLastError();
}
