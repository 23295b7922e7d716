// lt_team.h — threads that help with one job's results (lt_results.h); no HIP.
//
// None of them is needed: where a thread or memory for one cannot be had, those
// that are there, or the caller alone, do the work.
#pragma once
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <thread>
#include <utility>
#include <vector>

namespace lt {

// One result of a job: words of device memory and their place in the caller's.
struct OutSeg {
    uint32_t *dst;
    const uint32_t *src;
    uint64_t words;
};

// Threads that read each page of fresh pinned memory once, which maps it for the CPU
// (madvise does not take it), and map the pages of result buffers for writing,
// whose contents stay as they are (MADV_POPULATE_WRITE; a kernel without it leaves
// the faults to the copies).  Joined by wait() or with the object.
class PageMapper {
  public:
    ~PageMapper() { wait(); }
    // outs may be null.
    void start(const uint8_t *fresh, size_t fresh_bytes, const std::vector<OutSeg> *outs, uint32_t threads) {
        try {
            add((uintptr_t)fresh, (uintptr_t)fresh + fresh_bytes, kReadStep);
            reads = work.size();
            if (outs)
                for (const OutSeg &o : *outs)
                    add(((uintptr_t)o.dst + kAlign - 1) & ~(kAlign - 1),
                        ((uintptr_t)o.dst + 4 * o.words) & ~(kAlign - 1), kStep);
            for (uint32_t k = 0; k < threads; k++)
                team.emplace_back([this] {
                    for (size_t i; (i = next.fetch_add(1)) < work.size();)
                        if (!map(i)) return;
                });
        } catch (const std::exception &) {  // no more threads, or no memory for one
        }
    }
    // Ends it; the bytes of fresh memory that were read.
    size_t wait() {
        const size_t taken = next.exchange(work.size());  // the copies map the rest
        for (auto &t : team) t.join();
        team.clear();
        if (!ended)
            for (size_t i = 0; i < taken && i < reads; i++) bytes_read += work[i].second;
        ended = true;
        return bytes_read;
    }

  private:
    static constexpr uintptr_t kAlign = 4096, kStep = 1u << 20, kReadStep = 64u << 10;
    static constexpr int kPopulateWrite = 23;  // MADV_POPULATE_WRITE of Linux 5.14
    std::vector<std::pair<uintptr_t, size_t>> work;
    size_t reads = 0;  // of work, the first that are read
    size_t bytes_read = 0;
    bool ended = false;
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
    void start(uint32_t helpers) {  // once
        try {
            for (uint32_t k = 0; k < helpers; k++) team.emplace_back([this, k] { help(k + 1); });
        } catch (const std::exception &) {  // the team is smaller
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
    bool started = false, copying = false;
    PageMapper mapper;
    CopyTeam team;
    void start(const std::vector<OutSeg> &outs) {  // behind the job's first loads or launches
        started = true;
        const uint32_t readers = fresh_bytes ? help_most(1 + (fresh_bytes >> 19)) : 0;
        if (most || readers) mapper.start(fresh, fresh_bytes, most ? &outs : nullptr, std::max(most, readers));
    }
    CopyTeam &copiers() {  // one thread copies at about 32 GB/s, below the link's rate
        mapper.wait();
        if (!copying) team.start(most < 3 ? most : 3);
        copying = true;
        return team;
    }
};

}  // namespace lt
