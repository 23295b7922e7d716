// lt_kernels.h — walk, init and queue kernels (included by lt_engine.hip only).
//
// One walker per lane, kWpt walkers per thread.  A workgroup pass takes 1024
// walker records from the source queue (coalesced dwordx4 loads), walks each
// one while its vertex stays inside the span being processed, then appends
// the walkers that left to their destination partitions' queues:
//   1. LDS histogram of destination partitions (ds atomics, returns the rank
//      of the walker inside its bucket),
//   2. one global atomicAdd per (workgroup, destination) reserves a range of
//      queue slots, and an exclusive scan of the histogram gives each bucket
//      its place in an LDS staging buffer,
//   3. walkers are staged in LDS grouped by destination and written out by
//      consecutive lanes to consecutive queue slots.
// This is the two-level reshuffle of insertToQueueKernel
// (src/WalkManager.h:60-190) fused into the walk kernel
// (randomWalkKernel, src/WalkManager.h:229-246), so a residency costs one
// read and one write of the 16-byte record instead of two of each.
#pragma once
#include "lt_device.h"

namespace lt {

__device__ __forceinline__ uint32_t find_part(const Parts &pt, uint32_t v) {
    uint32_t p = pt.lut[v >> pt.lut_shift];
    while (v >= pt.node_off[p + 1]) ++p;
    return p;
}

__device__ __forceinline__ uint32_t load_agent(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Chunk k of partition part's queue: link a fresh chunk unless another lane
// linked one first (then return ours to the lost list).  Returns kEmpty if the
// pool is exhausted (flagged in ctl->overflow; the host turns it into an error).
__device__ uint32_t alloc_chunk(const Queues &q, uint32_t part, uint32_t k) {
    if (k >= q.maxc) {
        atomicOr(&q.ctl->overflow, 4u);
        return kEmpty;
    }
    uint32_t *slot = &q.frame[(size_t)part * q.maxc + k];
    const uint32_t top = q.ctl->top;
    const uint32_t i = atomicAdd(&q.ctl->popped, 1u);
    if (i >= top) {
        atomicOr(&q.ctl->overflow, 1u);
        return load_agent(slot);
    }
    const uint32_t c = q.free_stack[top - 1 - i];
    const uint32_t old = atomicCAS(slot, kEmpty, c);
    if (old == kEmpty) return c;
    const uint32_t j = atomicAdd(&q.ctl->nlost, 1u);
    if (j < kLostCap) q.lost[j] = c;
    else atomicOr(&q.ctl->overflow, 2u);
    return old;
}

// Chunk k of a queue whose first slot another workgroup reserved.  That
// workgroup took its slot range with an earlier atomicAdd, so it is running
// and links the chunk within a few microseconds: wait for the link (bounded),
// then link it ourselves if it still has not appeared.
__device__ __forceinline__ uint32_t get_chunk(const Queues &q, uint32_t part, uint32_t k) {
    if (k >= q.maxc) {
        atomicOr(&q.ctl->overflow, 4u);
        return kEmpty;
    }
    const uint32_t *slot = &q.frame[(size_t)part * q.maxc + k];
    uint32_t c = load_agent(slot);
    for (int it = 0; c == kEmpty && it < 4096; it++) {
        __builtin_amdgcn_s_sleep(4);
        c = load_agent(slot);
    }
    return c != kEmpty ? c : alloc_chunk(q, part, k);
}

// LDS layout of the append stage.  Every destination of a pass gets a slot:
// in direct mode the slot is the partition id (P slots); in hashed mode, for
// partition tables too large for that, the distinct destinations of the pass
// are numbered through an LDS hash table, so the layout depends only on the
// walkers per pass (at most one slot each).
constexpr uint32_t kDirectMaxP = 1024;  // larger partition tables use hashed slots
struct AppendLds {
    uint32_t *hist;   // [nslot] walkers per slot, then the slot's first reserved queue slot
    uint32_t *scan;   // [nslot+1] exclusive prefix of the walkers per slot
    uint32_t *ch0;    // [nslot] chunk holding the first reserved queue slot
    uint32_t *ch1;    // [nslot] chunk holding the last reserved queue slot
    uint32_t *part;   // hashed: [nslot] partition of each slot in use
    uint32_t *keys;   // hashed: [2*nslot] hash table of destination partitions (kEmpty = free)
    uint32_t *tslot;  // hashed: [2*nslot] slot given to each table entry
    uint32_t *nused;  // hashed: slots in use in the pass
    Walker *stage;    // [kBlock * wpt] walkers grouped by slot
    uint16_t *dst;    // [kBlock * wpt] slot of each staged walker
    uint32_t nslot;
    bool hashed;
};

// walkers staged per workgroup pass = kBlock * wpt
__host__ __device__ inline size_t append_lds_bytes(uint32_t P, int wpt) {
    const size_t nw = (size_t)kBlock * wpt;
    size_t b = P <= kDirectMaxP ? (4 * (size_t)P + 1) * 4 : (9 * nw + 2) * 4;
    b = (b + 15) & ~(size_t)15;
    return b + nw * (16 + 2);
}

__device__ __forceinline__ AppendLds carve_lds(uint8_t *smem, uint32_t P, int wpt) {
    AppendLds L;
    const uint32_t nw = kBlock * (uint32_t)wpt;
    L.hashed = P > kDirectMaxP;
    L.nslot = L.hashed ? nw : P;
    L.hist = (uint32_t *)smem;
    L.scan = L.hist + L.nslot;
    L.ch0 = L.scan + L.nslot + 1;
    L.ch1 = L.ch0 + L.nslot;
    L.part = L.ch1 + L.nslot;      // hashed mode only from here on
    L.keys = L.part + L.nslot;
    L.tslot = L.keys + 2 * L.nslot;
    L.nused = L.tslot + 2 * L.nslot;
    const size_t words = L.hashed ? 9 * (size_t)nw + 2 : 4 * (size_t)P + 1;
    const size_t off = (words * 4 + 15) & ~(size_t)15;
    L.stage = (Walker *)(smem + off);
    L.dst = (uint16_t *)(L.stage + nw);
    return L;
}

// Inclusive prefix sum over the 64 lanes of a wave with DPP moves: shifts by
// 1, 2, 4 and 8 within each row of 16 lanes (lanes shifted in from outside
// the row read 0), then row 0's total is added to row 1 and row 2's to row 3
// (row_bcast:15), then lane 31's sum to rows 2 and 3 (row_bcast:31).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);  // row_shr:1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true);  // row_shr:2
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, true);  // row_shr:4
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, true);  // row_shr:8
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false); // row_bcast:15, rows 1, 3
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false); // row_bcast:31, rows 2, 3
    return x;
}

// Exclusive scan of in[0..n) into out[], returns the total (all threads).
__device__ uint32_t block_exclusive_scan(const uint32_t *in, uint32_t *out, uint32_t n, uint32_t *s_wsum) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t per = (n + kBlock - 1) / kBlock;
    const uint32_t beg = min(tid * per, n), end = min(beg + per, n);
    uint32_t sum = 0;
    for (uint32_t i = beg; i < end; i++) sum += in[i];
    const uint32_t x = wave_incl_scan(sum);
    if (lane == 63) s_wsum[wave] = x;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kBlock / 64; w++) {
        const uint32_t s = s_wsum[w];
        before += (w < wave) ? s : 0u;
        total += s;
    }
    uint32_t run = before + x - sum;
    for (uint32_t i = beg; i < end; i++) {
        out[i] = run;
        run += in[i];
    }
    return total;
}

// Store walker w at position rank of slot sl's reservation (its first queue
// slot in L.hist[sl], the chunks it touches in L.ch0/L.ch1).
__device__ __forceinline__ void store_reserved(const Queues &q, const AppendLds &L, uint32_t sl, uint32_t rank,
                                               const Walker &w) {
    const uint32_t b = L.hist[sl];
    const uint32_t s = b + rank;
    const uint32_t c = (s >> kChunkLog2) == (b >> kChunkLog2) ? L.ch0[sl] : L.ch1[sl];
    if (c < q.nchunks) q.slab[(size_t)c * kChunk + (s & (kChunk - 1))] = w;
    else atomicOr(&q.ctl->overflow, 8u);
}

// One queue reservation per walker (append_mode 2).  Collective like
// block_append: every walker first takes its queue slot; the walkers whose
// slot starts a chunk link it, and after the barrier the others wait
// (bounded) for links made by reservations of other workgroups.
template <int WPT>
__device__ void append_one_level(const Queues &q, const Walker (&w)[WPT], const uint32_t (&dst)[WPT]) {
    uint32_t b[WPT], c[WPT];
#pragma unroll
    for (int k = 0; k < WPT; k++) {
        c[k] = kEmpty;
        if (dst[k] == kEmpty) continue;
        b[k] = atomicAdd(&qlen_of(q, dst[k]), 1u);
        if ((b[k] & (kChunk - 1)) == 0) c[k] = alloc_chunk(q, dst[k], b[k] >> kChunkLog2);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < WPT; k++) {
        if (dst[k] == kEmpty) continue;
        if ((b[k] & (kChunk - 1)) != 0) c[k] = get_chunk(q, dst[k], b[k] >> kChunkLog2);
        if (c[k] < q.nchunks) q.slab[(size_t)c[k] * kChunk + (b[k] & (kChunk - 1))] = w[k];
        else atomicOr(&q.ctl->overflow, 8u);
    }
    __syncthreads();
}

// block_append for partition tables above kDirectMaxP: the pass's distinct
// destinations are numbered through an open-addressed LDS table of
// 2 * nslot entries (at most nslot keys, so every probe sequence finds its
// key or a free entry), and the histogram, scan, reservations and staging of
// block_append then work on those slots instead of on partition ids.
template <int WPT>
__device__ void block_append_hashed(const Queues &q, const AppendLds &L, const Walker (&w)[WPT],
                                    const uint32_t (&dst)[WPT], uint32_t *s_wsum, int mode) {
    const uint32_t tid = threadIdx.x;
    const uint32_t T = 2 * L.nslot;  // a power of two
    for (uint32_t i = tid; i < T; i += kBlock) L.keys[i] = kEmpty;
    if (tid == 0) *L.nused = 0;
    __syncthreads();
    uint32_t ent[WPT] = {};
#pragma unroll
    for (int k = 0; k < WPT; k++) {
        if (dst[k] == kEmpty) continue;
        uint32_t h = dst[k] * 2654435761u;
        h = (h ^ (h >> 15)) & (T - 1);
        for (uint32_t probe = 0; probe < T; probe++) {
            const uint32_t old = atomicCAS(&L.keys[h], kEmpty, dst[k]);
            if (old == kEmpty || old == dst[k]) break;
            h = (h + 1) & (T - 1);
        }
        ent[k] = h;
    }
    __syncthreads();
    for (uint32_t i = tid; i < T; i += kBlock) {
        const uint32_t key = L.keys[i];
        if (key != kEmpty) {
            const uint32_t sidx = atomicAdd(L.nused, 1u);
            L.tslot[i] = sidx;
            L.part[sidx] = key;
            L.hist[sidx] = 0;
        }
    }
    __syncthreads();
    const uint32_t n = *L.nused;
    uint32_t sl[WPT], rank[WPT];
#pragma unroll
    for (int k = 0; k < WPT; k++) {
        sl[k] = dst[k] != kEmpty ? L.tslot[ent[k]] : kEmpty;
        if (dst[k] != kEmpty) rank[k] = atomicAdd(&L.hist[sl[k]], 1u);
    }
    __syncthreads();
    const uint32_t total = block_exclusive_scan(L.hist, L.scan, n, s_wsum);
    if (tid == 0) L.scan[n] = total;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += kBlock) {  // pass 1: the chunks this workgroup owns
        const uint32_t c = L.hist[i];
        if (c) {
            const uint32_t p = L.part[i];
            const uint32_t b = atomicAdd(&qlen_of(q, p), c);
            const uint32_t k0 = b >> kChunkLog2, k1 = (b + c - 1) >> kChunkLog2;
            const uint32_t c0 = (b & (kChunk - 1)) == 0 ? alloc_chunk(q, p, k0) : kEmpty;
            L.ch0[i] = c0;
            L.ch1[i] = k1 != k0 ? alloc_chunk(q, p, k1) : c0;
            L.hist[i] = b;
        }
    }
    for (uint32_t i = tid; i < n; i += kBlock) {  // pass 2: chunks owned by earlier reservations
        const uint32_t b = L.hist[i];
        if (L.scan[i + 1] != L.scan[i] && (b & (kChunk - 1)) != 0) {
            const uint32_t c0 = get_chunk(q, L.part[i], b >> kChunkLog2);
            const uint32_t k1 = (b + (L.scan[i + 1] - L.scan[i]) - 1) >> kChunkLog2;
            L.ch0[i] = c0;
            if (k1 == (b >> kChunkLog2)) L.ch1[i] = c0;
        }
    }
    __syncthreads();
    if (mode == 1) {  // uniform: each walker stored from its own lane
#pragma unroll
        for (int k = 0; k < WPT; k++)
            if (dst[k] != kEmpty) store_reserved(q, L, sl[k], rank[k], w[k]);
        __syncthreads();
        return;
    }
#pragma unroll
    for (int k = 0; k < WPT; k++) {
        if (dst[k] != kEmpty) {
            const uint32_t pos = L.scan[sl[k]] + rank[k];
            L.stage[pos] = w[k];
            L.dst[pos] = (uint16_t)sl[k];
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < total; i += kBlock) {
        const uint32_t slot = L.dst[i];
        const uint32_t b = L.hist[slot];
        const uint32_t s = b + (i - L.scan[slot]);
        const uint32_t c = (s >> kChunkLog2) == (b >> kChunkLog2) ? L.ch0[slot] : L.ch1[slot];
        if (c < q.nchunks) q.slab[(size_t)c * kChunk + (s & (kChunk - 1))] = L.stage[i];
        else atomicOr(&q.ctl->overflow, 8u);
    }
    __syncthreads();
}

// Append the walkers with dst[k] != kEmpty to their partitions' queues.
// Collective: every thread of the workgroup must call it.  Chunk ids are
// resolved once per (workgroup, destination): a reservation of at most
// kBlockWalkers <= kChunk slots touches at most two chunks; the range that
// contains a chunk's first slot links it, and a later range that arrives
// before that link is published links it itself (the CAS loser's chunk goes
// to the lost list).  Above kDirectMaxP partitions the slots are numbered
// through a hash table (block_append_hashed).
//
// hint: the chunk that held the end of partition threadIdx.x's queue when this
// thread last looked; a linked chunk stays linked for the launch, so one that
// is still the end's needs no lookup.
struct AppendHint {
    uint32_t k = kEmpty, c = kEmpty;  // chunk number in the queue, chunk id
    uint32_t len = 0;                 // first_hint's length of the queue, until second_hint
    bool look = false;
};

// First look, while the first walkers are fetched and walk (in two steps, so that
// neither load is waited for).  Only for launches of at most a workgroup per CU:
// those wait for every round trip, while in larger ones the lines, which every
// append writes, are better left alone.
__device__ __forceinline__ void first_hint(const Queues &q, uint32_t P, int mode, uint64_t passes, AppendHint &h) {
    h.look = passes <= 256 && P <= kDirectMaxP && mode != 2;
    if (h.look && threadIdx.x < P) h.len = load_agent(&qlen_of(q, threadIdx.x));
}

__device__ __forceinline__ void second_hint(const Queues &q, uint32_t P, AppendHint &h) {
    if (!h.look) return;  // uniform
    h.look = false;
    h.k = h.len >> kChunkLog2;
    if (threadIdx.x < P && h.k < q.maxc) h.c = load_agent(&q.frame[(size_t)threadIdx.x * q.maxc + h.k]);
}

//
// GEN: any partition count and append_mode; otherwise at most kDirectMaxP
// partitions and append_mode 0.
template <int WPT, bool GEN>
__device__ __forceinline__ void block_append(const Queues &q, uint32_t P, const AppendLds &L, const Walker (&w)[WPT],
                                             const uint32_t (&dst)[WPT], uint32_t *s_wsum, AppendHint &hint,
                                             int mode = 0) {
    if constexpr (GEN) {
        if (mode == 2) {  // uniform
            append_one_level<WPT>(q, w, dst);
            return;
        }
        if (L.hashed) {  // uniform: more partitions than LDS slots
            block_append_hashed<WPT>(q, L, w, dst, s_wsum, mode);
            return;
        }
    }
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < P; i += kBlock) L.hist[i] = 0;
    __syncthreads();
    uint32_t rank[WPT];
#pragma unroll
    for (int k = 0; k < WPT; k++)
        if (dst[k] != kEmpty) rank[k] = atomicAdd(&L.hist[dst[k]], 1u);
    __syncthreads();
    // The first reservation is on its way during the scan and the staging.
    uint32_t b0 = 0;
    if (tid < P && L.hist[tid]) b0 = atomicAdd(&qlen_of(q, tid), L.hist[tid]);
    const uint32_t total = block_exclusive_scan(L.hist, L.scan, P, s_wsum);
    if (tid == 0) L.scan[P] = total;
    __syncthreads();  // the scan reads hist segments that the loop below overwrites
    const bool staged = !(GEN && mode == 1);  // uniform; otherwise each walker is stored from its own lane
    if (staged) {
#pragma unroll
        for (int k = 0; k < WPT; k++) {
            if (dst[k] != kEmpty) {
                const uint32_t pos = L.scan[dst[k]] + rank[k];
                L.stage[pos] = w[k];
                L.dst[pos] = (uint16_t)dst[k];
            }
        }
    }
    // Pass 1: reserve and link the chunks this workgroup owns.  Pass 2 waits
    // for chunks owned by others only after every owned link is published,
    // so no owner ever waits before publishing.
    for (uint32_t i = tid; i < P; i += kBlock) {
        const uint32_t c = L.hist[i];
        if (c) {
            const uint32_t b = i == tid ? b0 : atomicAdd(&qlen_of(q, i), c);
            const uint32_t k0 = b >> kChunkLog2, k1 = (b + c - 1) >> kChunkLog2;
            const uint32_t c0 = (b & (kChunk - 1)) == 0 ? alloc_chunk(q, i, k0) : kEmpty;
            L.ch0[i] = c0;
            L.ch1[i] = k1 != k0 ? alloc_chunk(q, i, k1) : c0;
            L.hist[i] = b;
        }
    }
    for (uint32_t i = tid; i < P; i += kBlock) {
        const uint32_t b = L.hist[i];
        if (L.scan[i + 1] != L.scan[i]) {
            const uint32_t k0 = b >> kChunkLog2, k1 = (b + (L.scan[i + 1] - L.scan[i]) - 1) >> kChunkLog2;
            if ((b & (kChunk - 1)) != 0) {
                const uint32_t c0 = i == tid && k0 == hint.k && hint.c != kEmpty ? hint.c : get_chunk(q, i, k0);
                L.ch0[i] = c0;
                if (k1 == k0) L.ch1[i] = c0;
            }
            if (i == tid) {
                hint.k = k1;
                hint.c = L.ch1[i];
            }
        }
    }
    __syncthreads();
    if (!staged) {
#pragma unroll
        for (int k = 0; k < WPT; k++)
            if (dst[k] != kEmpty) store_reserved(q, L, dst[k], rank[k], w[k]);
        __syncthreads();
        return;
    }
    for (uint32_t i = tid; i < total; i += kBlock) {
        const uint32_t part = L.dst[i];
        const uint32_t b = L.hist[part];
        const uint32_t s = b + (i - L.scan[part]);
        const uint32_t c = (s >> kChunkLog2) == (b >> kChunkLog2) ? L.ch0[part] : L.ch1[part];
        if (c < q.nchunks) q.slab[(size_t)c * kChunk + (s & (kChunk - 1))] = L.stage[i];
        else atomicOr(&q.ctl->overflow, 8u);
    }
    __syncthreads();
}

// Per-thread event counts of one launch (far below 2^32), summed as u64.
struct Counters {
    uint32_t moves = 0, tele = 0, visits = 0, resid = 0, zc_moves = 0, zc_reads = 0;
    uint32_t *vbuf = nullptr, *vn = nullptr;  // workgroup visit buffer in LDS and its fill (walk kernels)
};

// Sum over the 64 lanes, in lane 63: 16 bits at a time, so that no 32-bit
// sum wraps.  (DPP moves: the six counters took 2 us of each launch's end by
// 64-bit shuffles.)
__device__ __forceinline__ unsigned long long wave_sum(uint32_t v) {
    const uint32_t lo = wave_incl_scan(v & 0xFFFFu), hi = wave_incl_scan(v >> 16);
    return (unsigned long long)lo + ((unsigned long long)hi << 16);
}

// Workgroup sum of the counters, added to slot blockIdx.x % kStatSlots, so
// that workgroups of one launch do not all update one cache line.
__device__ void flush_counters(const Counters &c, unsigned long long *stats) {
    __shared__ unsigned long long s_part[kBlock / 64][6];
    const uint32_t v[6] = {c.moves, c.tele, c.visits, c.resid, c.zc_moves, c.zc_reads};
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < 6; i++) {
        const unsigned long long x = wave_sum(v[i]);
        if (lane == 63) s_part[wave][i] = x;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        unsigned long long x = 0;
#pragma unroll
        for (int w = 0; w < kBlock / 64; w++) x += s_part[w][threadIdx.x];
        if (x) atomicAdd(&stats[(size_t)(blockIdx.x % kStatSlots) * kNumStats + threadIdx.x], x);
    }
}

// The graph span a walker is currently walking in.
struct Span {
    const uint64_t *rowptr;  // rowptr[v - nb] = global offset of v's first edge
    const uint32_t *col;     // col[e - eb], or the block headers of a packed slot
    const uint32_t *words;   // bit streams of a packed slot, nullptr for raw columns
    uint64_t eb;
    uint32_t nb, ne;
    int zc;
};

// Column of partition-local edge e.  A packed slot holds, per block of 16
// edges, {base, bit offset} (the next block's offset gives the width) and
// the bit streams: column = base + bits(offset + (e % 16) * width, width).
__device__ __forceinline__ uint32_t span_col(const Span &sp, uint64_t e) {
    if (!sp.words) return sp.col[e];
    const uint64_t k = e >> 4;
    const uint2 h = ((const uint2 *)sp.col)[k];
    const uint32_t w = (sp.col[2 * k + 3] - h.y) >> 4;
    const uint32_t pos = h.y + (uint32_t)(e & 15) * w;
    const uint32_t lo = sp.words[pos >> 5], hi = sp.words[(pos >> 5) + 1];
    const uint32_t bits = __builtin_amdgcn_alignbit(hi, lo, pos & 31u);
    return h.x + (w >= 32 ? bits : bits & ((1u << w) - 1u));
}

__device__ __forceinline__ uint64_t walker_id(const Walker &w) { return ((uint64_t)w.id_hi << 32) | w.id_lo; }

// Visits go to the visit log: a workgroup collects a pass's visits in LDS
// (consecutive lanes, one LDS atomic per wave) and copies them to its region of
// the log after the pass, in one reservation (walk_walkers).  Visits that do not
// fit the buffer are reserved in the log wave by wave, and those that do not fit
// the log, or of a job without one, are added to the counters directly.
constexpr uint32_t kVisitBuf = 4096;

__device__ __forceinline__ void count_direct(const AppArgs &a, uint32_t v) {
    atomicAdd(&a.counts[(size_t)(blockIdx.x % kCountCopies) * a.counts_stride + v], 1u);
}

// First of n entries reserved in the workgroup's region (vcap: past its end).
__device__ __forceinline__ uint32_t log_reserve(const AppArgs &a, uint32_t n) {
    const unsigned long long at = atomicAdd(&a.vcur[(blockIdx.x % kLogRegions) * kCurStride], (unsigned long long)n);
    return (uint32_t)min(at, (unsigned long long)a.vcap);
}

__device__ __forceinline__ uint32_t lanes_before(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ void log_store(const AppArgs &a, uint32_t i, uint32_t v) {
    if (i < a.vcap) a.vlog[(size_t)(blockIdx.x % kLogRegions) * a.vcap + i] = v;
    else count_direct(a, v);
}

__device__ __forceinline__ void count_visit(const AppArgs &a, uint32_t v, Counters &ct) {
    if (ct.vbuf) {
        const uint64_t m = __ballot(1);
        const uint32_t rank = lanes_before(m);
        uint32_t i = 0;
        if (rank == 0) i = atomicAdd(ct.vn, (uint32_t)__popcll(m));
        i = (uint32_t)__builtin_amdgcn_readfirstlane((int)i) + rank;
        if (i < kVisitBuf) {
            ct.vbuf[i] = v;
            return;
        }
        const uint64_t o = __ballot(1);
        const uint32_t orank = lanes_before(o);
        uint32_t j = 0;
        if (orank == 0) j = log_reserve(a, (uint32_t)__popcll(o));
        log_store(a, (uint32_t)__builtin_amdgcn_readfirstlane((int)j) + orank, v);
        return;
    }
    if (a.counts) count_direct(a, v);
}

// One update of app/pagerank.cu:26-44: count the visit, then teleport with
// probability 0.15 or move to a uniform neighbour.  A vertex without
// neighbours teleports (the reference divides by zero there).
__device__ __forceinline__ void step_pagerank(Walker &w, const Span &sp, const AppArgs &a, Counters &ct) {
    count_visit(a, w.cur, ct);
    ct.visits++;
    w.step -= 1;
    if (w.step == 0) return;
    const u32x4 x = draw(a.seed, walker_id(w), w.step, TAG_PAGERANK);
    bool tele = x.x < a.thresh;
    if (!tele) {
        const uint64_t *r = sp.rowptr + (w.cur - sp.nb);
        const uint64_t b = r[0], d = r[1] - b;
        if (d == 0) {
            tele = true;
            if (sp.zc) ct.zc_reads += a.rp_host;
        } else {
            w.cur = span_col(sp, b - sp.eb + bounded(x.y, x.z, d));
            ct.moves++;
            if (sp.zc) { ct.zc_moves++; ct.zc_reads += 1 + a.rp_host; }
        }
    }
    if (tele) {
        w.cur = (uint32_t)bounded(x.y, x.z, a.V);
        ct.tele++;
    }
}

// One update of app/ppr.cu:22-42: the endpoint is counted when one step is
// left; a vertex without neighbours is counted and ends the walk.
__device__ __forceinline__ void step_ppr(Walker &w, const Span &sp, const AppArgs &a, Counters &ct) {
    if (w.step == 1) {
        count_visit(a, w.cur, ct);
        ct.visits++;
    }
    w.step -= 1;
    if (w.step == 0) return;
    const uint64_t *r = sp.rowptr + (w.cur - sp.nb);
    const uint64_t b = r[0], d = r[1] - b;
    const u32x4 x = draw(a.seed, walker_id(w), w.step, TAG_PPR);  // (while r is fetched)
    if (d > 0) {
        w.cur = span_col(sp, b - sp.eb + bounded(x.y, x.z, d));
        ct.moves++;
        if (sp.zc) { ct.zc_moves++; ct.zc_reads += 1 + a.rp_host; }
    } else {
        count_visit(a, w.cur, ct);
        ct.visits++;
        w.step = 0;
        if (sp.zc) ct.zc_reads += a.rp_host;
    }
}

// One update of app/genericwalk.cu:22-32: a uniform neighbour move, or stop
// at a vertex without neighbours.  Records the number of moves made.
__device__ __forceinline__ void step_generic(Walker &w, const Span &sp, const AppArgs &a, Counters &ct) {
    const uint64_t *r = sp.rowptr + (w.cur - sp.nb);
    const uint64_t b = r[0], d = r[1] - b;
    uint32_t *path = a.paths ? a.paths + walker_id(w) * ((uint64_t)a.length + 1) : nullptr;
    if (path) path[a.length - w.step] = w.cur;  // the vertex after (length - step) moves
    const u32x4 x = draw(a.seed, walker_id(w), w.step, TAG_GENERIC);  // (while r is fetched)
    if (d > 0) {
        w.cur = span_col(sp, b - sp.eb + bounded(x.y, x.z, d));
        ct.moves++;
        if (sp.zc) { ct.zc_moves++; ct.zc_reads += 1 + a.rp_host; }
        w.step -= 1;
        if (w.step == 0) {
            if (a.moves_out) a.moves_out[walker_id(w)] = a.length;
            if (path) path[a.length] = w.cur;
        }
    } else {
        if (a.moves_out) a.moves_out[walker_id(w)] = a.length - w.step;
        w.step = 0;
        if (sp.zc) ct.zc_reads += a.rp_host;
    }
}

template <int APP>
__device__ __forceinline__ void app_step(Walker &w, const Span &sp, const AppArgs &a, Counters &ct) {
    if (APP == APP_PAGERANK) step_pagerank(w, sp, a, ct);
    else if (APP == APP_PPR) step_ppr(w, sp, a, ct);
    else step_generic(w, sp, a, ct);
}

__device__ __forceinline__ void finish_walker(const Walker &w, const AppArgs &a) {
    if (a.endpoints) a.endpoints[walker_id(w)] = w.cur;
}

__device__ __forceinline__ bool in_batch(const WalkArgs &a, uint32_t p) {
    bool in = false;
#pragma unroll
    for (uint32_t k = 0; k < kMaxZcBatch; k++) in |= a.srcs[k] == p;
    return in;
}

__device__ __forceinline__ void zerocopy_span(const WalkArgs &a, Span &sp) {
    sp.rowptr = a.ss.zc_rowptr + sp.nb;
    sp.col = a.ss.zc_col + sp.eb;
    sp.words = nullptr;
    sp.zc = 1;
}

// Puts what changed since the launch before, which comes with the arguments, into
// the record of partition p: a launch that sets two entries holds each round up
// for 7 us.
__device__ __forceinline__ void update_rec(const WalkArgs &a, uint32_t p, PartRec &r) {
    for (uint32_t k = 0; k < a.due.n; k++) {  // uniform
        if (a.due.part[k] == p) {
            r.rowptr = a.due.rowptr[k];
            r.col = a.due.col[k];
            r.words = a.due.words[k];
        }
    }
}

// Walk one residency; returns the destination partition or kEmpty when the
// walk is over.  With span_resident the walker continues into any partition
// whose slot is resident (and into the source slice itself, and into the others of
// a zero-copy batch).
//
// A launch lasts as long as its longest chain of steps, 50 us where the work
// of all lanes together is a few: a lane that leaves its span enters the next
// one in the turn in which the others step, rather than wait for all that stay
// (s20 ppr 15.9 -> 15.3 ms).  Where leaving the span ends the residency there is
// nothing to enter, and that loop stands by itself (14.7 ms; s20 reference rules
// as before, 1 % slower in the common loop).
template <int APP>
__device__ __forceinline__ uint32_t walk_residency(Walker &w, const WalkArgs &a, uint32_t src, const Span &src_sp,
                                                   Counters &ct) {
    if (!a.span_resident) {  // uniform
        while (w.step > 0 && w.cur - src_sp.nb < src_sp.ne - src_sp.nb) app_step<APP>(w, src_sp, a.app, ct);
        if (w.step > 0) return find_part(a.pt, w.cur);
        finish_walker(w, a.app);
        return kEmpty;
    }
    Span sp = src_sp;
    while (w.step > 0) {
        if ((w.cur - sp.nb) >= (sp.ne - sp.nb)) {
            uint32_t p = a.pt.lut[w.cur >> a.pt.lut_shift];
            PartRec r = a.pt.rec[p];
            while (w.cur >= r.ne) r = a.pt.rec[++p];
            update_rec(a, p, r);
            if (p == src) {
                sp = src_sp;
            } else {
                sp.nb = r.nb;
                sp.ne = r.ne;
                sp.eb = r.eb;
                if (r.rowptr) {
                    sp.rowptr = r.rowptr;
                    sp.col = r.col;
                    sp.words = r.words;
                    sp.zc = 0;
                } else {
                    if (!a.nsrc || !a.zerocopy || !in_batch(a, p)) return p;
                    zerocopy_span(a, sp);
                }
            }
        }
        app_step<APP>(w, sp, a.app, ct);
    }
    finish_walker(w, a.app);
    return kEmpty;
}

// One workgroup pass over nvalid <= kBlock * WPT walkers stored
// contiguously at cw: walk each, then append the survivors to their queues.
// The visit log is reserved before the append and written after it, so the
// reservation's round trip overlaps the append's own.
template <int APP, int WPT, bool GEN>
__device__ __forceinline__ void walk_walkers(const WalkArgs &a, const AppendLds &L, uint32_t *s_wsum, uint32_t src,
                                            const Span &src_sp, const Walker *cw, uint32_t nvalid, Counters &ct,
                                            AppendHint &hint) {
    Walker w[WPT];
    uint32_t dst[WPT];
#pragma unroll
    for (int k = 0; k < WPT; k++) {
        const uint32_t i = (uint32_t)k * kBlock + threadIdx.x;
        dst[k] = kEmpty;
        if (i < nvalid) {
            w[k] = cw[i];
            ct.resid++;
        } else {
            w[k].step = 0;
        }
    }
    second_hint(a.q, a.pt.P, hint);
#pragma unroll
    for (int k = 0; k < WPT; k++) {
        if ((uint32_t)k * kBlock + threadIdx.x < nvalid) dst[k] = walk_residency<APP>(w[k], a, src, src_sp, ct);
    }
    uint32_t n = 0, at = 0;
    if constexpr (APP != APP_GENERIC) {  // genericwalk counts no visits
        if (ct.vbuf) {  // uniform
            __syncthreads();
            n = min(*ct.vn, kVisitBuf);
            if (threadIdx.x == kBlock - 1 && n) at = log_reserve(a.app, n);
        }
    }
    block_append<WPT, GEN>(a.q, a.pt.P, L, w, dst, s_wsum, hint, a.append_mode);
    if constexpr (APP != APP_GENERIC) {
        if (ct.vbuf) {  // uniform
            __shared__ uint32_t s_at;
            if (threadIdx.x == kBlock - 1) {
                s_at = at;
                *ct.vn = 0;
            }
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < n; i += kBlock) log_store(a.app, s_at + i, ct.vbuf[i]);
            __syncthreads();
        }
    }
}

// WPT walkers per thread per pass (1, 2 or 4): small queues use 1 so that
// enough workgroups exist to fill the chip, large ones 4.  GEN: see block_append.
//
// A small launch waits for one round trip after another, and its code is
// one of them: every CU fetches what it runs.  So the source of a pass (a slice
// of one queue, queues of a batch, walkers in host memory, the device's
// choice) is picked in the loop and the pass itself stands here once, and
// what only large partition tables or append modes need is a kernel of its own.
template <int APP, int WPT, bool GEN>
__global__ __launch_bounds__(kBlock, WPT == 1 && !GEN ? 5 : 4) void walk_kernel(WalkArgs a) {
    constexpr int BW = kBlock * WPT;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ uint32_t s_wsum[kBlock / 64];
    // The arguments lie in memory: asked for one line at a time as the code gets
    // to them, each costs a small launch a round trip of its own.
    asm volatile("" ::"s"(a.app.seed), "s"(a.app.counts), "s"(a.app.vcur), "s"(a.app.rp_host), "s"(a.q.slab),
                 "s"(a.q.ctl), "s"(a.q.maxc), "s"(a.pt.node_off), "s"(a.pt.lut_shift), "s"(a.rowptr), "s"(a.src),
                 "s"(a.nhost), "s"(a.ss.ds));
    const AppendLds L = carve_lds(smem, a.pt.P, WPT);
    Counters ct;
    if constexpr (APP != APP_GENERIC) {
        __shared__ uint32_t s_vbuf[kVisitBuf], s_vn;
        if (a.app.vlog) {  // uniform
            if (threadIdx.x == 0) s_vn = 0;
            __syncthreads();
            ct.vbuf = s_vbuf;
            ct.vn = &s_vn;
        }
    }
    uint32_t src = a.src;
    Span sp;
    sp.rowptr = a.rowptr;
    sp.col = a.col;
    sp.words = a.words;
    sp.zc = a.zerocopy;
    sp.nb = a.nb;
    sp.ne = a.ne;
    sp.eb = a.eb;
    uint64_t lo = 0, hi;
    if (a.nsrc) {  // batch: the whole queues of several partitions, each in the partition table
        hi = a.voff[a.nsrc];
    } else if (a.nhost) {  // walkers of src spilled to host memory, read over PCIe
        hi = (uint64_t)a.nhost << kChunkLog2;
    } else if (a.ss.ds) {  // the decision of this iteration was taken on the device
        const DevSched &ds = *a.ss.ds;
        if (ds.choice < 0) return;
        src = (uint32_t)ds.choice;
        hi = ds.n;
        sp.rowptr = ds.rowptr;
        sp.col = ds.col;
        sp.words = ds.words;
        sp.zc = ds.zerocopy;
        sp.nb = ds.nb;
        sp.ne = ds.ne;
        sp.eb = ds.eb;
    } else {
        lo = (uint64_t)a.chunk_lo << kChunkLog2;
        hi = min((uint64_t)a.n, (uint64_t)a.chunk_hi << kChunkLog2);
    }
    if (lo + (uint64_t)blockIdx.x * BW >= hi) return;  // the device loop's grid is sized for any queue
    AppendHint hint;
    first_hint(a.q, a.pt.P, a.append_mode, (hi - lo) / BW, hint);
    // A pass: walkers [base, base + BW) clipped to n; base is a multiple of BW, so
    // it reads one chunk.
    for (uint64_t at = lo + (uint64_t)blockIdx.x * BW; at < hi; at += (uint64_t)gridDim.x * BW) {
        const Walker *cw;
        uint64_t base = at, n = hi;
        if (a.nhost) {
            const uint32_t k = (uint32_t)(at >> kChunkLog2);
            base = at & (kChunk - 1);
            n = a.hn[k];
            if (base >= n) continue;  // uniform per workgroup
            cw = a.hptr[k] + base;
        } else {
            if (a.nsrc) {
                uint32_t k = 0;
                while (k + 1 < a.nsrc && at >= a.voff[k + 1]) k++;
                src = a.srcs[k];
                base = at - a.voff[k];
                n = qlen_of(a.q, src);
                if (base >= n) continue;  // uniform per workgroup
                PartRec r = a.pt.rec[src];  // as a walker entering src reads it (walk_residency)
                update_rec(a, src, r);
                sp.rowptr = r.rowptr;
                sp.col = r.col;
                sp.words = r.words;
                sp.nb = r.nb;
                sp.ne = r.ne;
                sp.eb = r.eb;
                sp.zc = 0;
                if (a.zerocopy) zerocopy_span(a, sp);
            }
            const uint32_t chunk = a.q.frame[(size_t)src * a.q.maxc + (uint32_t)(base >> kChunkLog2)];
            if (chunk >= a.q.nchunks) {  // uniform per workgroup
                if (threadIdx.x == 0) atomicOr(&a.q.ctl->overflow, 8u);
                continue;
            }
            cw = a.q.slab + (size_t)chunk * kChunk + (uint32_t)(base & (kChunk - 1));
        }
        walk_walkers<APP, WPT, GEN>(a, L, s_wsum, src, sp, cw, (uint32_t)min(n - base, (uint64_t)BW), ct, hint);
    }
    flush_counters(ct, a.stats);
}

// PPR length (src/walk/SingleSource.h:12-17): 2 + number of draws that do not
// stop before the first one that does.
__device__ __forceinline__ uint32_t ppr_length(uint64_t seed, uint64_t id, uint32_t thresh) {
    uint32_t F = 0;
    for (uint32_t j = 0;; j++) {
        const u32x4 x = draw(seed, id, j, TAG_PPRLEN);
        if (x.x < thresh) return 2u + F;
        if (x.y < thresh) return 3u + F;
        if (x.z < thresh) return 4u + F;
        if (x.w < thresh) return 5u + F;
        F += 4;
        if (F > 0xFFFFFF00u) return 2u + F;
    }
}

// Create walkers [id_lo, id_hi) and append them to their start partitions'
// queues (GPUInitWalker::create + insertPushedToQueue, src/walk/InitWalk.h:16-20,
// src/WalkManager.h:341-350).
template <int APP>
__global__ __launch_bounds__(kBlock) void init_kernel(InitArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ uint32_t s_wsum[kBlock / 64];
    const AppendLds L = carve_lds(smem, a.pt.P, kWpt);
    AppendHint hint;
    for (uint64_t base = a.id_lo + (uint64_t)blockIdx.x * kBlockWalkers; base < a.id_hi;
         base += (uint64_t)gridDim.x * kBlockWalkers) {
        Walker w[kWpt];
        uint32_t dst[kWpt];
#pragma unroll
        for (int k = 0; k < kWpt; k++) {
            const uint64_t id = base + (uint64_t)k * kBlock + threadIdx.x;
            dst[k] = kEmpty;
            w[k].id_lo = (uint32_t)id;
            w[k].id_hi = (uint32_t)(id >> 32);
            if (id >= a.id_hi) {
                w[k].cur = 0;
                w[k].step = 0;
                continue;
            }
            if (APP == APP_PPR) {
                uint32_t src = a.app.source;
                if (a.app.q_off) {
                    uint32_t lo = 0, hi = a.app.nq;  // last query with q_off[q] <= id
                    while (hi - lo > 1) {
                        const uint32_t mid = (lo + hi) >> 1;
                        if (a.app.q_off[mid] <= id) lo = mid;
                        else hi = mid;
                    }
                    src = a.app.q_src[lo];
                }
                w[k].cur = src;
                w[k].step = ppr_length(a.app.seed, id, a.app.thresh);
            } else {
                const u32x4 x = draw(a.app.seed, id, 0, TAG_START);
                w[k].cur = (uint32_t)bounded(x.x, x.y, a.app.V);
                w[k].step = a.app.length;
            }
            if (w[k].step > 0) {
                dst[k] = find_part(a.pt, w[k].cur);
            } else {
                if (APP == APP_GENERIC && a.app.moves_out) a.app.moves_out[id] = 0;
                if (APP == APP_GENERIC && a.app.paths) a.app.paths[id * ((uint64_t)a.app.length + 1)] = w[k].cur;
                finish_walker(w[k], a.app);
            }
        }
        block_append<kWpt, true>(a.q, a.pt.P, L, w, dst, s_wsum, hint);
    }
}

// Written through to the host.
__device__ __forceinline__ void to_host(uint32_t *p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The queue lengths, PoolCtl and the log's cursors go to q.packed for the host
// (Engine::wait_meta), each word with the launch's number beside it: the host
// takes a word once its number is there, and no lane has to wait for the link to
// take all others' words before one says that they are there (1.3 us).
__device__ __forceinline__ void tell_host(const Queues &q, uint32_t i, uint32_t v) {
    __hip_atomic_store(&q.packed[i], (uint64_t)q.seq << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ uint32_t log_fill(const Queues &q, uint32_t r) {
    return (uint32_t)min(q.vcur[r * kCurStride], 0xFFFFFFFFull);
}

// Collective over one workgroup; runs after every queue update of the stream.
__device__ void pack_meta(const Queues &q) {
    for (uint32_t i = threadIdx.x; i < q.P; i += blockDim.x) tell_host(q, i, qlen_of(q, i));
    if (threadIdx.x < sizeof(PoolCtl) / 4) tell_host(q, q.P + threadIdx.x, ((const uint32_t *)q.ctl)[threadIdx.x]);
    if (q.vcur && threadIdx.x < kLogRegions) tell_host(q, q.P + 4 + threadIdx.x, log_fill(q, threadIdx.x));
}

__global__ __launch_bounds__(kBlock) void pack_meta_kernel(Queues q) { pack_meta(q); }

template <uint32_t N>
__device__ __forceinline__ void set_entries(PartRec *rec, const TableEntries<N> &b) {
    const uint32_t k = threadIdx.x;
    if (k < b.n) {
        PartRec *r = &rec[b.part[k]];
        r->rowptr = b.rowptr[k];
        r->col = b.col[k];
        r->words = b.words[k];
    }
}

// Return the popped-but-unused state of the pool, the lost chunks and the
// consumed source chunks to the free stack; clear the source queues after their
// last slice; tell the host the queue lengths.  One workgroup, for all sources of
// a batch's launch.
//
// Every round of a job waits for this kernel, a chain of round trips: what it
// reads by known addresses is read at once, and the host, which needs the
// lengths only, gets them before the chunks move (its next walk is behind this
// kernel in the stream).
__global__ __launch_bounds__(kBlock) void fixup_kernel(Queues q, Consumed d, PartRec *rec) {
    __shared__ uint32_t s_top, s_nlost, s_off[kMaxZcBatch + 1];
    const uint32_t tid = threadIdx.x;
    const uint32_t n = d.n, lo = d.chunk_lo;
    const PoolCtl c = *q.ctl;
    const uint32_t len = tid < q.P ? qlen_of(q, tid) : 0u;
    const uint32_t fill = q.vcur && tid < kLogRegions ? log_fill(q, tid) : 0u;
    if (tid < n) {
        const uint32_t nch = (qlen_of(q, d.src[tid]) + kChunk - 1) >> kChunkLog2;
        const uint32_t hi = min(d.chunk_hi, nch);
        s_off[tid + 1] = hi > lo ? hi - lo : 0;
    }
    __syncthreads();
    if (tid == 0) {
        const uint32_t popped = min(c.popped, c.top);
        const uint32_t nlost = c.nlost < kLostCap ? c.nlost : kLostCap;
        PoolCtl after{c.top - popped, 0, 0, c.overflow};
        s_off[0] = 0;
        for (uint32_t k = 0; k < n; k++) s_off[k + 1] += s_off[k];
        s_top = after.top;
        s_nlost = nlost;
        if (after.top + nlost + s_off[n] > q.nchunks) {
            after.overflow |= 16u;
            s_nlost = 0;
            for (uint32_t k = 0; k <= n; k++) s_off[k] = 0;
        }
        after.top += s_nlost + s_off[n];
        *q.ctl = after;
        tell_host(q, q.P, after.top);
        tell_host(q, q.P + 1, 0);
        tell_host(q, q.P + 2, 0);
        tell_host(q, q.P + 3, after.overflow);
    }
    for (uint32_t i = tid; i < q.P; i += kBlock) {
        uint32_t v = i == tid ? len : qlen_of(q, i);
#pragma unroll
        for (uint32_t k = 0; k < kMaxZcBatch; k++) v = d.last && k < n && d.src[k] == i ? 0u : v;
        tell_host(q, i, v);
    }
    if (q.vcur && tid < kLogRegions) tell_host(q, q.P + 4 + tid, fill);
    __syncthreads();
    const uint32_t top = s_top, nlost = s_nlost, cnt = s_off[n];
    for (uint32_t i = tid; i < nlost; i += kBlock) q.free_stack[top + i] = q.lost[i];
    uint32_t k = 0;
    for (uint32_t j = tid; j < cnt; j += kBlock) {
        while (j >= s_off[k + 1]) k++;
        uint32_t *f = &q.frame[(size_t)d.src[k] * q.maxc + lo + (j - s_off[k])];
        q.free_stack[top + nlost + j] = *f;
        *f = kEmpty;
    }
    if (tid < n && d.last) qlen_of(q, d.src[tid]) = 0;
    set_entries(rec, d.due);
}

// Copy the queues of a spill round into host memory: walker i of partition
// k goes to slot hstart[k] + i of its host chunks (vector stores over PCIe).
__global__ __launch_bounds__(256) void spill_gather_kernel(SpillArgs s) {
    const uint64_t total = s.prefix[s.nv];
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
        uint32_t lo = 0, hi = s.nv;  // last k with prefix[k] <= idx
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s.prefix[mid] <= idx) lo = mid;
            else hi = mid;
        }
        const uint64_t i = idx - s.prefix[lo];
        const uint32_t c = s.q.frame[(size_t)s.part[lo] * s.q.maxc + (uint32_t)(i >> kChunkLog2)];
        if (c >= s.q.nchunks) {
            atomicOr(&s.q.ctl->overflow, 8u);
            continue;
        }
        const uint64_t hp = s.hstart[lo] + i;
        s.hptr[s.hbase[lo] + (uint32_t)(hp >> kChunkLog2)][hp & (kChunk - 1)] =
            s.q.slab[(size_t)c * kChunk + (i & (kChunk - 1))];
    }
}

// Return the spilled partitions' chunks to the free stack and empty their
// queues; pack the queue lengths.  One workgroup, after spill_gather_kernel.
__global__ __launch_bounds__(kBlock) void release_queues_kernel(SpillArgs s) {
    __shared__ uint32_t s_top;
    if (threadIdx.x == 0) {
        s_top = s.q.ctl->top;
        if (s_top + s.cprefix[s.nv] > s.q.nchunks) {
            s.q.ctl->overflow |= 16u;
            s_top = 0xFFFFFFFFu;
        }
    }
    __syncthreads();
    const uint32_t top = s_top;
    if (top != 0xFFFFFFFFu) {
        for (uint32_t k = 0; k < s.nv; k++) {
            const uint32_t nch = s.cprefix[k + 1] - s.cprefix[k];
            uint32_t *f = s.q.frame + (size_t)s.part[k] * s.q.maxc;
            for (uint32_t j = threadIdx.x; j < nch; j += blockDim.x) {
                s.q.free_stack[top + s.cprefix[k] + j] = f[j];
                f[j] = kEmpty;
            }
        }
        for (uint32_t k = threadIdx.x; k < s.nv; k += blockDim.x) qlen_of(s.q, s.part[k]) = 0;
    }
    __syncthreads();
    if (threadIdx.x == 0 && top != 0xFFFFFFFFu) s.q.ctl->top = top + s.cprefix[s.nv];
    __syncthreads();
    pack_meta(s.q);
}

// Empty every queue and put all chunks on the free stack.
__global__ void reset_queues_kernel(Queues q, uint32_t P) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = tid; i < (size_t)P * q.maxc; i += stride) q.frame[i] = kEmpty;
    for (size_t i = tid; i < q.nchunks; i += stride) q.free_stack[i] = (uint32_t)i;
    for (size_t i = tid; i < (size_t)P * kQStride; i += stride) q.qlen[i] = 0;
    if (tid == 0) {
        q.ctl->top = q.nchunks;
        q.ctl->popped = 0;
        q.ctl->nlost = 0;
        q.ctl->overflow = 0;
    }
}

// Partition table updates, all those due before a walk in one launch.
__global__ void set_tables_kernel(PartRec *rec, TableBatch b) { set_entries(rec, b); }

// Copy of a partition's two slices from mapped host memory (or HBM) into a cache
// slot, 4-byte words: 64 workgroups with eight loads per lane in flight fill
// the link.
struct PullArgs {
    const uint32_t *src[2];
    uint32_t *dst[2];
    uint64_t words[2];
};

__device__ __forceinline__ void pull_words(const uint32_t *src, uint32_t *dst, uint64_t n) {
    constexpr int kAhead = 8;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + (kAhead - 1) * stride < n; i += kAhead * stride) {
        uint32_t v[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; k++) v[k] = __builtin_nontemporal_load(&src[i + k * stride]);
#pragma unroll
        for (int k = 0; k < kAhead; k++) dst[i + k * stride] = v[k];
    }
    for (; i < n; i += stride) dst[i] = __builtin_nontemporal_load(&src[i]);
}

__global__ __launch_bounds__(256) void pull_kernel(PullArgs a) {
#pragma unroll
    for (int s = 0; s < 2; s++) pull_words(a.src[s], a.dst[s], a.words[s]);
}

// Plain streaming copy of n 16-byte vectors (known HBM traffic: 16n read, 16n written).
__global__ __launch_bounds__(256) void copy_probe_kernel(const uint4 *src, uint4 *dst, uint64_t n) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// counts[v] = sum over the kCountCopies copies of v's count (in place into copy 0).
__global__ __launch_bounds__(256) void sum_count_copies_kernel(uint32_t *counts, uint32_t V) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += stride) {
        uint32_t s = 0;
#pragma unroll
        for (uint32_t c = 0; c < kCountCopies; c++) s += counts[c * (size_t)V + v];
        counts[v] = s;
    }
}

__global__ void fill_u32_kernel(uint32_t *p, size_t n, uint32_t v) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t i = tid; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// ---- device-side scheduling ------------------------------------------------
// Lowest / highest value of the workgroup.
template <bool MAX>
__device__ __forceinline__ unsigned long long block_extreme(unsigned long long v, unsigned long long *s_wave) {
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(v, off, 64);
        v = (MAX ? o > v : o < v) ? o : v;
    }
    if ((threadIdx.x & 63u) == 0) s_wave[threadIdx.x >> 6] = v;
    __syncthreads();
    for (int w = 0; w < kBlock / 64; w++) {
        const unsigned long long o = s_wave[w];
        v = (MAX ? o > v : o < v) ? o : v;
    }
    return v;
}

// What decide_kernel may need to know of a partition.
struct PartState {
    uint32_t len = 0, nb = 0, ne = 0, resident = 0;
    uint64_t eb = 0, ee = 0;
    int32_t slot = -1;
    const uint32_t *words = nullptr;
};

__device__ __forceinline__ PartState part_state(const Queues &q, const SchedState &ss, const Parts &pt, uint32_t p) {
    PartState o;
    o.len = qlen_of(q, p);
    const PartRec r = pt.rec[p];
    o.nb = r.nb;
    o.ne = r.ne;
    o.eb = r.eb;
    o.words = r.words;
    o.ee = pt.edge_off[p + 1];
    o.resident = ss.resident[p];
    o.slot = ss.slot_of[p];
    return o;
}

// One workgroup ends the iteration before (its queue's chunks, the popped and the
// lost ones go back to the free stack, as in fixup_kernel) and decides the next
// with the plain rules: the partition with the most queued walkers (lowest id
// on ties); walk it in place if resident, read it over PCIe if it holds fewer
// than zc_threshold walkers, else copy it into a free slot or into the slot of
// the resident partition with the fewest walkers.  Tables are updated here; the
// copy is done by load_kernel next.
//
// Nothing but round trips: every thread reads its own partition's state at
// once, so that the one whose partition is chosen holds all that the copy and the
// walk need, and these read one record instead of looking it up.
__global__ __launch_bounds__(kBlock) void decide_kernel(Queues q, SchedState ss, Parts pt, BlockImages bi) {
    __shared__ unsigned long long s_wave[3][kBlock / 64];
    __shared__ uint32_t s_prev, s_resident;
    const uint32_t tid = threadIdx.x, P = pt.P;
    DevSched d = *ss.ds;
    const PoolCtl ctl = *q.ctl;
    PartState own;
    if (tid < P) own = part_state(q, ss, pt, tid);
    const int32_t in_slot = tid < ss.nslots ? ss.part_in_slot[tid] : 0;
    const int32_t prev = d.choice;
    unsigned long long best = 0;
    for (uint32_t p = tid; p < P; p += kBlock) {
        const unsigned long long c = p == tid ? own.len : qlen_of(q, p);
        if ((int32_t)p == prev) {
            s_prev = (uint32_t)c;
        } else if (c) {
            const unsigned long long key = (c << 32) | (0xFFFFFFFFull - p);
            best = key > best ? key : best;
        }
    }
    best = block_extreme<true>(best, s_wave[0]);
    if (prev >= 0) {
        uint32_t nch = (s_prev + kChunk - 1) >> kChunkLog2, nlost = min(ctl.nlost, kLostCap);
        const uint32_t top = ctl.top - min(ctl.popped, ctl.top);
        PoolCtl after{top, 0, 0, ctl.overflow};
        if (top + nlost + nch > q.nchunks) {
            after.overflow |= 16u;
            nlost = nch = 0;
        }
        for (uint32_t i = tid; i < nlost; i += kBlock) q.free_stack[top + i] = q.lost[i];
        for (uint32_t j = tid; j < nch; j += kBlock) {
            uint32_t *f = &q.frame[(size_t)prev * q.maxc + j];
            q.free_stack[top + nlost + j] = *f;
            *f = kEmpty;
        }
        if (tid == 0) {
            after.top += nlost + nch;
            *q.ctl = after;
            qlen_of(q, (uint32_t)prev) = 0;
        }
    }
    d.load = 0;
    d.zerocopy = 0;
    if (best == 0) {
        if (tid == 0) {
            d.choice = -1;
            *ss.ds = d;
        }
        return;
    }
    const uint32_t c = 0xFFFFFFFFu - (uint32_t)(best & 0xFFFFFFFFull);
    const bool chosen = tid == c % kBlock;
    if (chosen) {
        if (c != tid) own = part_state(q, ss, pt, c);
        s_resident = own.resident;
    }
    __syncthreads();
    const bool need_slot = !s_resident && (best >> 32) >= ss.zc_threshold;
    unsigned long long free_slot = ~0ull, victim = ~0ull;
    if (need_slot) {
        for (uint32_t s = tid; s < ss.nslots; s += kBlock)
            if ((s == tid ? in_slot : ss.part_in_slot[s]) < 0 && s < free_slot) free_slot = s;
        for (uint32_t p = tid; p < P; p += kBlock) {
            // (the chosen thread's own state may be another partition's by now)
            const bool mine = p == tid && !chosen;
            if (p == c || !(mine ? own.resident : ss.resident[p])) continue;
            const unsigned long long len = (int32_t)p == prev ? 0 : mine ? own.len : qlen_of(q, p);
            const unsigned long long key = (len << 32) | p;
            victim = key < victim ? key : victim;
        }
        free_slot = block_extreme<false>(free_slot, s_wave[1]);
        victim = block_extreme<false>(victim, s_wave[2]);
    }
    if (!chosen) return;
    const uint64_t n1 = (uint64_t)own.ne - own.nb + 1, m = own.ee - own.eb;
    d.choice = (int32_t)c;
    d.iterations++;
    d.n = own.len;
    d.nb = own.nb;
    d.ne = own.ne;
    d.eb = own.eb;
    int32_t slot = own.slot;
    if (!own.resident) {
        if (!need_slot || (free_slot == ~0ull && victim == ~0ull)) {  // few walkers, or nothing to evict
            d.zerocopy = 1;
            d.zc_calls++;
            d.rowptr = ss.zc_rowptr + own.nb;
            d.col = ss.zc_col + own.eb;
            d.words = nullptr;
            *ss.ds = d;
            return;
        }
        slot = (int32_t)free_slot;
        if (free_slot == ~0ull) {
            const uint32_t v = (uint32_t)(victim & 0xFFFFFFFFull);
            slot = ss.slot_of[v];
            ss.slot_of[v] = -1;
            ss.resident[v] = 0;
            ss.rec[v].rowptr = nullptr;
        }
    }
    uint8_t *base = ss.slots + (size_t)slot * ss.slot_bytes;
    d.rowptr = (const uint64_t *)base;
    d.col = (const uint32_t *)(base + n1 * 8);
    d.words = own.words;
    if (!own.resident) {
        const uint64_t img = bi.img ? bi.size[c] : 0;  // block image bytes, 0 = raw columns
        d.words = img ? d.col + 2 * ((m + kBlockEdges - 1) / kBlockEdges + 1) : nullptr;
        ss.slot_of[c] = slot;
        ss.part_in_slot[slot] = (int32_t)c;
        ss.resident[c] = 1;
        ss.rec[c].rowptr = d.rowptr;
        ss.rec[c].col = d.col;
        ss.rec[c].words = d.words;
        d.load = 1;
        d.from[0] = (const uint32_t *)(ss.zc_rowptr + own.nb);
        d.from[1] = img ? (const uint32_t *)(bi.img + bi.off[c]) : ss.zc_col + own.eb;
        d.count[0] = 2 * n1;
        d.count[1] = img ? img / 4 : m;
        d.loads++;
        d.h2d_bytes += n1 * 8 * ss.rp_host + (img ? img : m * 4);
    }
    *ss.ds = d;
}

// Copy the decided partition from pinned host memory into its slot: rowptr
// slice, then the col slice or (block slots) the partition's block image.
__global__ __launch_bounds__(256) void load_kernel(const DevSched *ds) {
    if (!ds->load) return;
    pull_words(ds->from[0], (uint32_t *)ds->rowptr, ds->count[0]);
    pull_words(ds->from[1], (uint32_t *)ds->col, ds->count[1]);
}

// Columns of a block image, in edge order: a lane an edge, so a block's header and
// words are read by neighbouring lanes at once.  Bound by the link that the image
// comes over (55 GB/s), not by this.
__global__ __launch_bounds__(256) void unblock_kernel(const uint32_t *__restrict__ img, uint64_t m,
                                                      uint32_t *__restrict__ col) {
    Span sp{};
    sp.col = img;
    sp.words = img + 2 * ((m + kBlockEdges - 1) / kBlockEdges + 1);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m; e += stride) col[e] = span_col(sp, e);
}

// Unpacks a packed partition image into the col slice of an HBM slot whose
// rowptr slice is already in place (it gives the row boundaries; rowptr[0] is
// the partition's first global edge).  Image layout: meta u32[2*nch] (nch =
// ceil(m/64); per chunk its first word and the codes of its four 16-edge
// blocks), bit streams u32[nwords] + 2 zero words; an anchor (first edge of
// its row or of its chunk, or any edge of a block coded 255) holds the column
// in vbits bits, any other edge the gap to the previous column in its block's
// width.  The bytes written equal the raw col slice.
//
// One wave per kUnpackChunks consecutive 64-edge chunks, one lane per edge:
//   - the row holding the wave's first edge comes from a 64-ary search of
//     rowptr (one ballot per level); later chunks carry it forward;
//   - whether a lane's edge starts a row: rows ending inside the chunk are
//     read 64 at a time (coalesced) and mark their end in the wave's LDS
//     flags;
//   - each lane's bit offset: exclusive scan of the field widths; the chunk's
//     words (at most 64) sit one per lane and are fetched by shuffle;
//   - columns: inclusive scan of the fields minus the scan just before the
//     lane's anchor (u32 arithmetic; the difference is exact);
//   - the 64 columns of a chunk are stored by consecutive lanes.
constexpr uint32_t kUnpackChunks = 8;

__global__ __launch_bounds__(256) void unpack_kernel(const uint8_t *__restrict__ img, uint32_t n, uint64_t m,
                                                     uint64_t nwords, uint32_t vbits,
                                                     const uint64_t *__restrict__ rowptr,
                                                     uint32_t *__restrict__ col) {
    const uint64_t nch = (m + 63) / 64;
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint64_t cb = wave * kUnpackChunks;
    if (cb >= nch) return;  // whole wave
    const uint64_t ce = cb + kUnpackChunks < nch ? cb + kUnpackChunks : nch;
    const uint64_t eb = rowptr[0];
    const uint32_t *meta = (const uint32_t *)img;
    const uint32_t *wd = meta + 2 * nch;
    __shared__ uint8_t s_starts[4][64];  // per wave: chunk edges that start a row
    volatile uint8_t *starts = s_starts[threadIdx.x >> 6];

    // row r0 holding edge 64*cb: the last r < n with rowptr[r] - eb <= 64*cb
    uint64_t e0 = cb * 64;
    uint32_t lo = 0, hi = n - 1;
    while (hi > lo) {
        const uint64_t span = (uint64_t)hi - lo + 1;
        const uint32_t idx = lo + (uint32_t)(span * lane / 64);
        const uint64_t mask = __ballot(rowptr[idx] - eb <= e0);
        const uint32_t k = (uint32_t)__popcll(mask) - 1;  // lane 0 (idx = lo) always holds
        const uint32_t nlo = __shfl(idx, k, 64);
        const uint32_t nxt = __shfl(idx, k < 63 ? k + 1 : 63, 64);
        hi = k < 63 ? nxt - 1 : hi;
        lo = nlo;
        if (hi < lo) hi = lo;
    }
    uint32_t r0 = lo;

    for (uint64_t c = cb; c < ce; c++) {
        e0 = c * 64;
        const uint32_t cnt = (uint32_t)(m - e0 < 64 ? m - e0 : 64);
        // the chunk's words, one per lane, and its block codes
        const uint64_t w_beg = meta[2 * c], w_end = c + 1 < nch ? meta[2 * c + 2] : nwords;
        const uint32_t bw = (meta[2 * c + 1] >> ((lane >> 4) * 8)) & 0xFFu;
        const uint32_t word = w_beg + lane < w_end ? wd[w_beg + lane] : 0u;
        // rows r0+1.. that end inside the chunk: a row ending at chunk edge i
        // means edge i starts a row; mark those edges in the wave's LDS flags
        uint32_t adv = 0;
        starts[lane] = 0;
        for (uint32_t base = r0 + 1;; base += 64) {
            const uint32_t idx = base + lane;
            const uint64_t end = idx <= n ? rowptr[idx] - eb : ~0ull;  // > e0 for every idx > r0
            const uint32_t p = (uint32_t)(end - e0 < 65 ? end - e0 : 65);  // 1..65
            if (p < 64) starts[p] = 1;
            const uint32_t p63 = (uint32_t)__builtin_amdgcn_readlane((int)p, 63);
            adv += (uint32_t)__popcll(__ballot(p <= 64));
            if (p63 > 64 || base + 64 > n) break;
        }
        const bool valid = lane < cnt;
        const bool anchor = valid && (lane == 0 || starts[lane] || bw == 0xFFu);
        const uint32_t len = valid ? (anchor ? vbits : bw) : 0u;
        const uint32_t pos = wave_incl_scan(len) - len;
        const uint32_t wi = pos >> 5;
        const uint32_t lo_w = __shfl(word, wi, 64);
        const uint32_t hi_w = __shfl(word, (wi + 1) & 63u, 64);
        // bits [pos, pos + len) of the chunk: (hi:lo) >> (pos % 32), low len bits
        const uint32_t bits = __builtin_amdgcn_alignbit(wi + 1 < 64 ? hi_w : 0u, lo_w, pos & 31u);
        const uint32_t v = len >= 32 ? bits : bits & ((1u << len) - 1u);
        const uint32_t incl = wave_incl_scan(v);
        const uint64_t heads = __ballot(anchor) & (lane == 63 ? ~0ull : ((2ull << lane) - 1));
        const uint32_t head = 63u - (uint32_t)__clzll(heads);  // lane 0 is always a head
        const uint32_t before = __shfl(incl, head > 0 ? head - 1 : 0, 64);
        if (valid) col[e0 + lane] = incl - (head > 0 ? before : 0u);
        r0 += adv;
    }
}

}  // namespace lt
