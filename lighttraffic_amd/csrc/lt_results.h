// lt_results.h — results from the device to the caller's memory (included by
// lt_engine.hip only).
//
// The caller's buffers are ordinary host memory.  hipMemcpy into them ran at
// 14-17 GB/s (20 MB of fresh pages: 1.5 ms, as long as the walk that made
// them).  Results of up to 256 KB are written to pinned memory by the job's last
// kernels.  Larger ones go through a ring of pinned buffers, which kernels of
// the compute stream fill at the link's rate (50 GB/s) while a few threads copy
// another one out.  (Copies on a second stream overlap the walk only when HIP
// gives the two streams hardware queues of their own, which it did not for the
// second engine of a process; then they took twice as long as these.)  Fixed-
// length walks over the flat arrays write their endpoints to the ring themselves.
// Other threads have fresh pages of the caller's mapped, and read those of a new
// ring for the first time, while the job walks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lt_kernels.h"
#include "lt_team.h"

namespace lt {

// Results small enough to be written to pinned memory by a kernel.
constexpr uint64_t kSmallOut = 64 * 1024;  // words
constexpr uint32_t kOutSegs = 4;
struct SmallOut {
    uint32_t n;
    const uint32_t *src[kOutSegs];
    uint32_t end[kOutSegs];  // words of the segments up to and including k
    uint32_t *dst;           // pinned, mapped
};

__global__ __launch_bounds__(256) void small_out_kernel(SmallOut o) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    uint32_t k = 0, beg = 0;
    while (k < o.n && i >= o.end[k]) beg = o.end[k++];
    if (k < o.n) to_host(&o.dst[i], o.src[k][i - beg]);
}

// n words to a ring buffer, both 16-byte aligned.  64 workgroups fill the link.
__global__ __launch_bounds__(256) void fill_ring_kernel(const uint32_t *src, uint32_t *dst, uint64_t n) {
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = tid; i < n / 4; i += stride) ((uint4 *)dst)[i] = ((const uint4 *)src)[i];
    if (tid < n % 4) dst[n / 4 * 4 + tid] = src[n / 4 * 4 + tid];
    __threadfence_system();
}

// A sequence number for the host, behind what the stream's kernels wrote to it.
__global__ void mark_kernel(uint32_t *flag, uint32_t seq) {
    __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The job's event counters summed over their slots into pinned memory, then the
// sequence number that the host polls.  One workgroup, last of the job.
__global__ __launch_bounds__(kStatSlots) void finish_kernel(const unsigned long long *stats, uint32_t *out,
                                                            uint32_t *flag, uint32_t seq) {
    __shared__ unsigned long long s_part[kStatSlots / 64][kNumStats];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < kNumStats; i++) {
        unsigned long long x = stats[(size_t)threadIdx.x * kNumStats + i];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if (lane == 0) s_part[wave][i] = x;
    }
    __syncthreads();
    if (threadIdx.x < kNumStats) {
        unsigned long long x = 0;
#pragma unroll
        for (uint32_t w = 0; w < kStatSlots / 64; w++) x += s_part[w][threadIdx.x];
        to_host(&out[2 * threadIdx.x], (uint32_t)x);
        to_host(&out[2 * threadIdx.x + 1], (uint32_t)(x >> 32));
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Clears what a job accumulates into: counters of visits and events, the visit
// log's cursors.
__global__ __launch_bounds__(256) void begin_kernel(uint32_t *counts, uint64_t n, unsigned long long *stats,
                                                    unsigned long long *vcur) {
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = tid; i < n / 4; i += stride) ((uint4 *)counts)[i] = make_uint4(0, 0, 0, 0);
    if (tid < n % 4) counts[n / 4 * 4 + tid] = 0;
    for (uint64_t i = tid; i < (uint64_t)kNumStats * kStatSlots; i += stride) stats[i] = 0;
    if (vcur && tid < kLogRegions) vcur[tid * kCurStride] = 0;
}

}  // namespace lt
