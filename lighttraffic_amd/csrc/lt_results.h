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
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <system_error>
#include <thread>
#include <utility>
#include <vector>

#include "lt_kernels.h"

namespace lt {

// One result of a job: words of device memory and their place in the caller's.
struct OutSeg {
    uint32_t *dst;
    const uint32_t *src;
    uint64_t words;
};

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

// Threads that read each page of fresh pinned memory once, which maps it for the CPU
// (madvise does not take it), and map the pages of result buffers for writing,
// whose contents stay as they are (MADV_POPULATE_WRITE; a kernel without it leaves
// the faults to the copies).  Joined by wait() or with the object.
class PageMapper {
  public:
    ~PageMapper() { wait(); }
    void start(const uint8_t *fresh, size_t fresh_bytes, const std::vector<OutSeg> &outs, uint32_t threads) {
        add((uintptr_t)fresh, (uintptr_t)fresh + fresh_bytes, kReadStep);
        reads = work.size();
        for (const OutSeg &o : outs)
            add(((uintptr_t)o.dst + kAlign - 1) & ~(kAlign - 1), ((uintptr_t)o.dst + 4 * o.words) & ~(kAlign - 1),
                kStep);
        try {
            for (uint32_t k = 0; k < threads; k++)
                team.emplace_back([this] {
                    for (size_t i; (i = next.fetch_add(1)) < work.size();)
                        if (!map(i)) return;
                });
        } catch (const std::system_error &) {
        }
    }
    void wait() {
        next.store(work.size());  // the copies map the rest
        for (auto &t : team) t.join();
        team.clear();
    }

  private:
    static constexpr uintptr_t kAlign = 4096, kStep = 1u << 20, kReadStep = 64u << 10;
    static constexpr int kPopulateWrite = 23;  // MADV_POPULATE_WRITE of Linux 5.14
    std::vector<std::pair<uintptr_t, size_t>> work;
    size_t reads = 0;  // of work, the first that are read
    std::atomic<size_t> next{0};
    std::vector<std::thread> team;

    void add(uintptr_t lo, uintptr_t hi, uintptr_t step) {
        for (uintptr_t at = lo; at < hi; at += step) work.push_back({at, hi - at < step ? hi - at : step});
    }
    bool map(size_t i) {
        const auto &w = work[i];
        if (i >= reads) return madvise((void *)w.first, w.second, kPopulateWrite) == 0;
        for (uintptr_t at = w.first; at < w.first + w.second; at += kAlign) (void)*(volatile const uint8_t *)at;
        return true;
    }
};

// A few threads that copy one block of memory at a time, each its share, and
// end with the object.
class CopyTeam {
  public:
    explicit CopyTeam(uint32_t helpers) {
        try {
            for (uint32_t k = 0; k < helpers; k++) team.emplace_back([this, k] { help(k + 1); });
        } catch (const std::system_error &) {  // no more threads: the team is smaller
        }
    }
    ~CopyTeam() {
        stop = true;
        turn.fetch_add(1, std::memory_order_release);
        for (auto &t : team) t.join();
    }
    void copy(void *d, const void *s, size_t bytes) {
        dst = (uint8_t *)d;
        src = (const uint8_t *)s;
        n = bytes;
        parts = team.size() + 1;
        done.store(0, std::memory_order_relaxed);
        turn.fetch_add(1, std::memory_order_release);
        share(0);
        while (done.load(std::memory_order_acquire) != team.size()) __builtin_ia32_pause();
    }

  private:
    std::vector<std::thread> team;
    std::atomic<uint32_t> turn{0}, done{0};
    bool stop = false;
    uint8_t *dst = nullptr;
    const uint8_t *src = nullptr;
    size_t n = 0, parts = 1;

    void share(size_t k) {  // on page boundaries of the block
        const size_t per = ((n + parts - 1) / parts + 4095) & ~(size_t)4095;
        const size_t lo = k * per < n ? k * per : n, hi = lo + per < n ? lo + per : n;
        if (hi > lo) memcpy(dst + lo, src + lo, hi - lo);
    }
    void help(size_t k) {
        for (uint32_t seen = 0;;) {
            uint32_t t;
            for (uint32_t spins = 0; (t = turn.load(std::memory_order_acquire)) == seen; spins++) {
                if (spins < 4096) __builtin_ia32_pause();
                else std::this_thread::yield();
            }
            seen = t;
            if (stop) return;
            share(k);
            done.fetch_add(1, std::memory_order_release);
        }
    }
};

// At most `wanted` threads beside the caller's, and 4.  (The system is asked once: 20 us.)
inline uint32_t help_most(size_t wanted) {
    static const uint32_t cpus = std::max(1u, std::thread::hardware_concurrency());
    return (uint32_t)std::min<size_t>({wanted, 4, cpus - 1});
}

// Threads that help with one job's results: none for small ones.
struct ResultHelpers {
    uint32_t most = 0;
    const uint8_t *fresh = nullptr;  // pinned memory that the CPU has not read yet
    size_t fresh_bytes = 0;
    bool started = false;
    PageMapper mapper;
    std::unique_ptr<CopyTeam> team;
    void start(const std::vector<OutSeg> &outs) {  // behind the job's first loads or launches
        started = true;
        const uint32_t readers = fresh_bytes ? help_most(1 + (fresh_bytes >> 19)) : 0;
        if (most || readers) mapper.start(fresh, fresh_bytes, most ? outs : std::vector<OutSeg>(), std::max(most, readers));
    }
    CopyTeam &copiers() {  // one thread copies at about 32 GB/s, below the link's rate
        mapper.wait();
        if (!team) team.reset(new CopyTeam(most < 3 ? most : 3));
        return *team;
    }
};

}  // namespace lt
