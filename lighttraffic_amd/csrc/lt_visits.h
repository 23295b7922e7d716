// lt_visits.h — visit counting through a log (included by lt_kernels.h).
//
// Random u32 atomics on global memory run at 27 G/s on this card, whatever
// the footprint, scope or number of copies (5 G/s on a thousand addresses), so
// a walk that counts every vertex it visits with one is bound by them: 1.8 of
// the 2.8 ms of a pagerank job of 48 M visits.  Walks therefore write the
// visited vertices to a log (streaming stores) and the log is counted in LDS:
//   visit_tile_kernel     histogram of each 16 K-entry tile over bins of 32 K vertices
//   visit_scan_kernel     place of each (bin, tile) run, bin totals
//   visit_scatter_kernel  tiles partitioned by bin: the low 15 bits of each
//                         entry, as u16, in runs
//   visit_hist_kernel     one workgroup per unit (64 K entries or more) of a bin:
//                         counters in LDS, written out as a partial histogram
//   visit_sum_kernel      counts[v] += the partial histograms of v's bin
// With at most kFewBins bins the hist kernel reads the log itself, once per
// bin, and the first three are left out.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lt {

constexpr uint32_t kBinLog2 = 15;
constexpr uint32_t kBin = 1u << kBinLog2;  // vertices per bin: 128 KB of LDS counters
constexpr uint32_t kMaxBins = 2048;
constexpr uint32_t kFewBins = 4;
constexpr uint32_t kVisitThreads = 1024;
constexpr uint32_t kTile = 16 * kVisitThreads;  // log entries partitioned by one workgroup
constexpr uint32_t kHistUnit = 1u << 16;        // entries of a bin counted by one workgroup, at least
constexpr uint32_t kHistUnits = 512;            // units a log is cut into, at most (and one a bin more)
constexpr uint32_t kFewUnits = 1024;            // tiles times bins counted without a sort, at most
constexpr uint32_t kLogRegions = 8;  // one per XCD: workgroup b appends to region b % 8
constexpr uint32_t kRepl = 4;        // copies of a tile's histogram: R-MAT visits crowd into few
                                     // bins, and lanes that add to one address take turns

// A log of visited vertices: region r holds min(cur[r * kCurStride], cap) entries
// at log + r * cap (a cursor counts the entries that found no room too, so it has
// 64 bits).  With n > 0 it is one run of n entries instead.
constexpr uint32_t kCurStride = 16;  // one cursor per 128-byte line
struct VisitLog {
    uint32_t *log;
    unsigned long long *cur;
    uint32_t cap;
    uint32_t n;
    uint32_t tiles;  // tiles per region (of the run)
};

// Scratch of a count (see the kernels).
struct VisitScratch {
    uint16_t *sorted;    // [entries]
    uint32_t *run;       // [nbins][tiles of all regions]
    uint32_t *total;     // [nbins]
    uint32_t *unit_off;  // [nbins + 1]
    uint32_t *partial;   // [units][kBin]
    uint32_t unit;       // entries per unit
};

// Entries of tile t: base pointer and number.
__device__ __forceinline__ uint32_t tile_of(const VisitLog &l, uint32_t t, const uint32_t *&p) {
    const uint32_t r = t / l.tiles, i = t - r * l.tiles;
    const uint32_t n = l.n ? l.n : (uint32_t)min(l.cur[r * kCurStride], (unsigned long long)l.cap);
    const uint64_t at = (uint64_t)i * kTile;
    p = l.log + (size_t)r * l.cap + at;
    return at < n ? (uint32_t)min((uint64_t)kTile, n - at) : 0u;
}

// Exclusive scan over n <= 2 * kVisitThreads values of LDS (in place), returns
// the total.  Collective over kVisitThreads threads.
__device__ __forceinline__ uint32_t scan_lds(uint32_t *v, uint32_t n, uint32_t *s_w) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t i0 = 2 * tid, a = i0 < n ? v[i0] : 0u, b = i0 + 1 < n ? v[i0 + 1] : 0u;
    uint32_t x = a + b;
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < kVisitThreads / 64; w++) {
        before += w < wave ? s_w[w] : 0u;
        all += s_w[w];
    }
    const uint32_t ex = before + x - a - b;
    if (i0 < n) v[i0] = ex;
    if (i0 + 1 < n) v[i0 + 1] = ex + a;
    __syncthreads();
    return all;
}

__global__ __launch_bounds__(kVisitThreads) void visit_tile_kernel(VisitLog l, VisitScratch s, uint32_t nbins,
                                                                   uint32_t ntiles) {
    extern __shared__ uint32_t s_hist[];  // [kRepl][nbins]
    const uint32_t *p;
    const uint32_t n = tile_of(l, blockIdx.x, p);
    for (uint32_t i = threadIdx.x; i < kRepl * nbins; i += kVisitThreads) s_hist[i] = 0;
    __syncthreads();
    uint32_t *h = s_hist + (threadIdx.x & (kRepl - 1)) * nbins;
    if (n == kTile) {
        uint4 v[kTile / kVisitThreads / 4];
#pragma unroll
        for (uint32_t k = 0; k < kTile / kVisitThreads / 4; k++) v[k] = ((const uint4 *)p)[k * kVisitThreads + threadIdx.x];
#pragma unroll
        for (uint32_t k = 0; k < kTile / kVisitThreads / 4; k++) {
            atomicAdd(&h[v[k].x >> kBinLog2], 1u);
            atomicAdd(&h[v[k].y >> kBinLog2], 1u);
            atomicAdd(&h[v[k].z >> kBinLog2], 1u);
            atomicAdd(&h[v[k].w >> kBinLog2], 1u);
        }
    } else {
        for (uint32_t i = threadIdx.x; i < n; i += kVisitThreads) atomicAdd(&h[p[i] >> kBinLog2], 1u);
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < nbins; b += kVisitThreads) {
        uint32_t c = 0;
#pragma unroll
        for (uint32_t r = 0; r < kRepl; r++) c += s_hist[r * nbins + b];
        s.run[(size_t)b * ntiles + blockIdx.x] = c;
    }
}

// One workgroup per bin: run lengths over the tiles -> run starts within the
// bin, and the bin's total.
__global__ __launch_bounds__(kVisitThreads) void visit_scan_kernel(VisitScratch s, uint32_t ntiles) {
    __shared__ uint32_t s_v[2 * kVisitThreads], s_w[kVisitThreads / 64];
    uint32_t *run = s.run + (size_t)blockIdx.x * ntiles;
    uint32_t sum = 0;
    for (uint32_t t0 = 0; t0 < ntiles; t0 += 2 * kVisitThreads) {
        const uint32_t m = min(2 * kVisitThreads, ntiles - t0);
        for (uint32_t i = threadIdx.x; i < m; i += kVisitThreads) s_v[i] = run[t0 + i];
        __syncthreads();
        const uint32_t all = scan_lds(s_v, m, s_w);
        for (uint32_t i = threadIdx.x; i < m; i += kVisitThreads) run[t0 + i] = sum + s_v[i];
        sum += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) s.total[blockIdx.x] = sum;
}

// Partition one tile by bin: ranks from LDS histograms (kRepl per bin), entries
// staged in LDS in bin order, runs written by consecutive lanes.
__host__ __device__ inline size_t scatter_lds(uint32_t nbins) {
    return 4 * ((size_t)(kRepl + 1) * nbins) + 4 * (size_t)kTile;
}
__global__ __launch_bounds__(kVisitThreads) void visit_scatter_kernel(VisitLog l, VisitScratch s, uint32_t nbins,
                                                                      uint32_t ntiles) {
    constexpr uint32_t kPer = kTile / kVisitThreads;
    extern __shared__ uint32_t s_mem[];
    __shared__ uint32_t s_w[kVisitThreads / 64];
    uint32_t *hist = s_mem;                // [nbins][kRepl], then the start of each
    uint32_t *dst = hist + kRepl * nbins;  // [nbins] bin starts in sorted[], then minus the staged start
    uint32_t *stage = dst + nbins;         // [kTile] bin << 16 | low bits
    const uint32_t *p;
    const uint32_t n = tile_of(l, blockIdx.x, p);
    if (n == 0) return;
    const uint32_t tid = threadIdx.x;
    uint32_t v[kPer], rank[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
        const uint32_t i = k * kVisitThreads + tid;
        v[k] = i < n ? p[i] : 0u;
    }
    for (uint32_t i = tid; i < kRepl * nbins; i += kVisitThreads) hist[i] = 0;
    for (uint32_t i = tid; i < nbins; i += kVisitThreads) dst[i] = s.total[i];
    __syncthreads();
    scan_lds(dst, nbins, s_w);
    const uint32_t rep = tid & (kRepl - 1);
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++)
        if (k * kVisitThreads + tid < n) rank[k] = atomicAdd(&hist[(v[k] >> kBinLog2) * kRepl + rep], 1u);
    __syncthreads();
    // starts of the (bin, replica) runs in the stage, 2 * kVisitThreads at a time
    uint32_t before = 0;
    for (uint32_t i0 = 0; i0 < kRepl * nbins; i0 += 2 * kVisitThreads) {
        const uint32_t m = min(2 * kVisitThreads, kRepl * nbins - i0);
        const uint32_t all = scan_lds(hist + i0, m, s_w);
        if (before)
            for (uint32_t i = tid; i < m; i += kVisitThreads) hist[i0 + i] += before;
        before += all;
        __syncthreads();
    }
    for (uint32_t b = tid; b < nbins; b += kVisitThreads)
        dst[b] += s.run[(size_t)b * ntiles + blockIdx.x] - hist[b * kRepl];
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++)
        if (k * kVisitThreads + tid < n) {
            const uint32_t b = v[k] >> kBinLog2;
            stage[hist[b * kRepl + rep] + rank[k]] = b << 16 | (v[k] & (kBin - 1));
        }
    __syncthreads();
    for (uint32_t i = tid; i < n; i += kVisitThreads) {
        const uint32_t e = stage[i];
        s.sorted[dst[e >> 16] + i] = (uint16_t)e;
    }
}

// Partial histogram of one unit.  SORTED: unit u counts a piece of a
// bin's entries (units are numbered bin by bin); else unit u = bin * ntiles +
// tile counts the entries of that bin in tile `tile` of the log.
template <bool SORTED>
__global__ __launch_bounds__(kVisitThreads) void visit_hist_kernel(VisitLog l, VisitScratch s, uint32_t nbins,
                                                                   uint32_t ntiles) {
    __shared__ uint32_t s_cnt[kBin];
    const uint32_t tid = threadIdx.x;
    if constexpr (SORTED) {
        __shared__ uint32_t s_w[kVisitThreads / 64], s_bin, s_beg, s_len;
        uint32_t *first = s_cnt, *unit = s_cnt + kMaxBins;  // bins' first entries and first units
        for (uint32_t b = tid; b < nbins; b += kVisitThreads) {
            first[b] = s.total[b];
            unit[b] = (first[b] + s.unit - 1) / s.unit;
        }
        if (tid == 0) s_bin = kMaxBins;
        __syncthreads();
        const uint32_t entries = scan_lds(first, nbins, s_w), units = scan_lds(unit, nbins, s_w);
        for (uint32_t b = tid; b < nbins; b += kVisitThreads) {
            const uint32_t u0 = unit[b], u1 = b + 1 < nbins ? unit[b + 1] : units;
            const uint32_t end = b + 1 < nbins ? first[b + 1] : entries;
            if (blockIdx.x >= u0 && blockIdx.x < u1) {
                s_bin = b;
                s_beg = first[b] + (blockIdx.x - u0) * s.unit;
                s_len = min(s.unit, end - s_beg);
            }
            if (blockIdx.x == 0) {
                s.unit_off[b] = u0;
                if (b + 1 == nbins) s.unit_off[nbins] = units;
            }
        }
        __syncthreads();
        if (s_bin == kMaxBins) return;  // uniform: fewer units than workgroups
        const uint32_t beg = s_beg, len = s_len;
        __syncthreads();
        for (uint32_t i = tid; i < kBin; i += kVisitThreads) s_cnt[i] = 0;
        __syncthreads();
        const uint16_t *e = s.sorted + beg;
        uint32_t i = tid;
        for (; i + 7 * kVisitThreads < len; i += 8 * kVisitThreads) {
            uint32_t x[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; k++) x[k] = e[i + k * kVisitThreads];
#pragma unroll
            for (uint32_t k = 0; k < 8; k++) atomicAdd(&s_cnt[x[k]], 1u);
        }
        for (; i < len; i += kVisitThreads) atomicAdd(&s_cnt[e[i]], 1u);
    } else {
        const uint32_t bin = blockIdx.x / ntiles;
        const uint32_t *p;
        const uint32_t n = tile_of(l, blockIdx.x - bin * ntiles, p);
        for (uint32_t i = tid; i < kBin; i += kVisitThreads) s_cnt[i] = 0;
        if (blockIdx.x == 0 && tid <= nbins) s.unit_off[tid] = tid * ntiles;
        __syncthreads();
        for (uint32_t i = tid; i < n; i += kVisitThreads) {
            const uint32_t x = p[i];
            if (x >> kBinLog2 == bin) atomicAdd(&s_cnt[x & (kBin - 1)], 1u);
        }
    }
    __syncthreads();
    uint4 *out = (uint4 *)(s.partial + (size_t)blockIdx.x * kBin);
    for (uint32_t i = tid; i < kBin / 4; i += kVisitThreads) out[i] = ((const uint4 *)s_cnt)[i];
}

// counts[v] += v's partial counts; the log is empty afterwards.
__global__ __launch_bounds__(256) void visit_sum_kernel(VisitLog l, VisitScratch s, uint32_t *counts, uint32_t V) {
    const uint32_t v = blockIdx.x * 256 + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < kLogRegions && l.cur) l.cur[threadIdx.x * kCurStride] = 0;
    if (v >= V) return;
    const uint32_t b = v >> kBinLog2;
    const uint32_t u0 = s.unit_off[b], u1 = s.unit_off[b + 1];
    const uint32_t *q = s.partial + (size_t)u0 * kBin + (v & (kBin - 1));
    uint32_t c = 0, u = u0;
    for (; u + 8 <= u1; u += 8, q += 8 * kBin) {  // eight loads in flight: a hot bin has hundreds of units
        uint32_t x[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) x[k] = q[k * kBin];
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) c += x[k];
    }
    for (; u < u1; u++, q += kBin) c += *q;
    if (c) counts[v] += c;
}

}  // namespace lt
