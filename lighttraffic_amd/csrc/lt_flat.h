// lt_flat.h — walks of a graph that lies whole in HBM (included by lt_engine.hip only).
//
// With every partition cached and raw, the slots are slices of one rowptr and
// one col array, so a walker needs neither a partition lookup nor a queue: a
// lane creates a walker, walks it to its end and takes the next one.
#pragma once
#include "lt_kernels.h"

namespace lt {

struct FlatArgs {
    AppArgs app;
    const uint32_t *rowptr;  // [V+1]
    const uint32_t *col;
    uint64_t id_lo, id_hi;  // walkers of the launch
    unsigned long long *stats;
};

__global__ __launch_bounds__(256) void narrow_rowptr_kernel(const uint64_t *rp, uint32_t *out, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = (uint32_t)rp[i];
}

// bounded(hi, lo, n) for n < 2^32: floor((hi * 2^32 + lo) * n / 2^64) =
// floor((hi * n + floor(lo * n / 2^32)) / 2^32), two 32-bit products.
__device__ __forceinline__ uint32_t bounded32(uint32_t hi, uint32_t lo, uint32_t n) {
    const uint64_t t = ((uint64_t)lo * n) >> 32;
    return (uint32_t)(((uint64_t)hi * n + t) >> 32);
}

// Row of v: first edge and degree.
__device__ __forceinline__ void row_of(const uint32_t *rp, uint32_t v, uint32_t &b, uint32_t &d) {
    b = rp[v];
    d = rp[(size_t)v + 1] - b;
}

// Edges are read at uniformly random places of an array far larger than the
// caches, rows at places that follow the degrees: the non-temporal hint keeps
// the rows in L2.
__device__ __forceinline__ uint32_t load_col(const uint32_t *p) { return __builtin_nontemporal_load(p); }

// Fixed-length walks (pagerank, genericwalk), one walker per lane.
//
// Bound: lines missed in L2.  On this card random reads that miss L2 run at 55 G
// lines/s whatever the footprint (64 MB to 8 GB) and however many waves or
// loads per lane are in flight; L2 hits run at 250 G/s.  A move misses at
// least its edge's line, and its row's when the row is not hot.  R-MAT s22
// ef16 genericwalk (4.8 M walkers, 48 M moves, 0.5 GB of columns): 1.11 ms, 43 G
// moves/s, 0.79 of that rate; through the queues 1.44 ms and 0.2 ms of
// creating the walkers and clearing the queues.  4 to 8 workgroups per CU and 1, 2 or
// 4 walkers per lane in lockstep measured the same.
template <int APP>
__global__ __launch_bounds__(kBlock) void flat_walk_kernel(FlatArgs a) {
    const uint32_t *rp = a.rowptr;
    const uint64_t seed = a.app.seed;
    const uint32_t length = a.app.length;
    Counters ct;
    const uint64_t n = a.id_hi - a.id_lo;
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t id = a.id_lo + (uint64_t)blockIdx.x * kBlock + threadIdx.x; id < a.id_hi; id += stride) {
        const u32x4 s = draw(seed, id, 0, TAG_START);
        uint32_t cur = bounded32(s.x, s.y, a.app.V);
        ct.resid += length > 0;
        uint32_t left = length;
        if constexpr (APP == APP_PAGERANK) {
            for (; left > 0; left--) {
                // the draw does not wait for the vertex being read
                const u32x4 x = draw(seed, id, left - 1, TAG_PAGERANK);
                // every walker visits `length` vertices: its place in the log is known
                if (a.app.vlog) __builtin_nontemporal_store(cur, &a.app.vlog[(length - left) * n + (id - a.id_lo)]);
                else if (a.app.counts) count_direct(a.app, cur);
                ct.visits++;
                if (left == 1) break;
                uint32_t b = 0, d = 0;
                if (x.x >= a.app.thresh) row_of(rp, cur, b, d);
                if (d == 0) {  // teleport, also from a vertex without neighbours
                    cur = bounded32(x.y, x.z, a.app.V);
                    ct.tele++;
                } else {
                    cur = load_col(a.col + b + bounded32(x.y, x.z, d));
                    ct.moves++;
                }
            }
        } else {
            uint32_t *path = a.app.paths ? a.app.paths + id * ((uint64_t)length + 1) : nullptr;
            for (; left > 0; left--) {
                const u32x4 x = draw(seed, id, left, TAG_GENERIC);
                uint32_t b, d;
                row_of(rp, cur, b, d);
                if (path) path[length - left] = cur;
                if (d == 0) break;
                cur = load_col(a.col + b + bounded32(x.y, x.z, d));
                ct.moves++;
            }
            if (path) {
                if (left == 0) path[length] = cur;
                for (uint32_t i = length - left + 1; left > 0 && i <= length; i++) path[i] = 0xFFFFFFFFu;
            }
            if (a.app.moves_out) a.app.moves_out[id] = length - left;
        }
        if (a.app.endpoints) a.app.endpoints[id] = cur;
    }
    flush_counters(ct, a.stats);
}

// PPR walks have geometric lengths: a workgroup owns a range of walkers and a
// lane takes the next one as soon as its walk ends, so lanes idle only at the
// end of the range (a wave that waits for its longest walk keeps about a
// quarter of its lanes busy at p = 0.15).
__global__ __launch_bounds__(kBlock) void flat_ppr_kernel(FlatArgs a) {
    const uint32_t *rp = a.rowptr;
    Counters ct;
    __shared__ uint32_t s_next;
    const uint64_t n = a.id_hi - a.id_lo, per = (n + gridDim.x - 1) / gridDim.x;
    const uint64_t lo = a.id_lo + (uint64_t)blockIdx.x * per;
    const uint32_t mine = lo < a.id_hi ? (uint32_t)min(per, a.id_hi - lo) : 0u;
    if (threadIdx.x == 0) s_next = kBlock;
    __syncthreads();
    uint32_t q = 0;  // query of the lane's walker; walker ids only grow
    uint32_t cur = 0, step = 0;
    uint64_t id = 0;
    const auto start = [&](uint32_t i) {
        id = lo + i;
        cur = a.app.source;
        if (a.app.q_off) {
            if (id >= a.app.q_off[q + 1]) {
                uint32_t l = q + 1, h = a.app.nq;  // last query with q_off[q] <= id
                while (h - l > 1) {
                    const uint32_t mid = (l + h) >> 1;
                    if (a.app.q_off[mid] <= id) l = mid;
                    else h = mid;
                }
                q = l;
            }
            cur = a.app.q_src[q];
        }
        step = ppr_length(a.app.seed, id, a.app.thresh);
        ct.resid++;
    };
    uint32_t i = threadIdx.x;
    if (i < mine) start(i);
    while (i < mine) {  // one step, or one walk's end, per turn
        bool over = --step == 0;
        if (!over) {
            const u32x4 x = draw(a.app.seed, id, step, TAG_PPR);
            uint32_t b, d;
            row_of(rp, cur, b, d);
            if (d == 0) {
                over = true;
            } else {
                cur = load_col(a.col + b + bounded32(x.y, x.z, d));
                ct.moves++;
            }
        }
        if (over) {
            if (a.app.vlog) a.app.vlog[id - a.id_lo] = cur;  // one visit per walker
            else if (a.app.counts) count_direct(a.app, cur);
            ct.visits++;
            if (a.app.endpoints) a.app.endpoints[id] = cur;
            i = atomicAdd(&s_next, 1u);
            if (i < mine) start(i);
        }
    }
    flush_counters(ct, a.stats);
}

}  // namespace lt
