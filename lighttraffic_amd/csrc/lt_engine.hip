// lt_engine.hip — the GPU engine behind lt_engine_* / lt_run_*.
//
// Host side of the hot path: the HBM partition cache (role of GPUGraph,
// src/GraphLoader.h:160-240), the walker queues (GPUListPool,
// src/buffer/Pool.h:530-646), the per-partition processing step
// (GPUWalkManager::processInMemory, src/WalkManager.h:362-404) and the plain
// scheduler loop (GPUScheduler / Scheduler, src/Scheduler.h:13-454).
#include <hip/hip_runtime.h>

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <deque>
#include <memory>
#include <vector>

#include "lt_internal.h"
#include "lt_kernels.h"
#include "lt_flat.h"
#include "lt_mlp.h"
#include "lt_results.h"
#include "lt_sched.h"

#define LT_HIP(call)                                                                                   \
    do {                                                                                               \
        hipError_t _e = (call);                                                                        \
        if (_e != hipSuccess) {                                                                        \
            lt::set_error("%s:%d %s: %s", __FILE__, __LINE__, #call, hipGetErrorString(_e));            \
            return LT_E_HIP;                                                                           \
        }                                                                                              \
    } while (0)

#define LT_TRY(expr)                    \
    do {                                \
        lt_status _s = (expr);          \
        if (_s != LT_OK) return _s;     \
    } while (0)

namespace lt {

// Reference page size (numBlock * threadPerBlock * walkerPerThread,
// src/Type.h:10-14): the "full queue" threshold of getComputedPartition.
constexpr uint64_t kRefPage = 82ull * 512 * 4;

template <typename T>
static lt_status dmalloc(T **p, size_t count) {
    *p = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc((void **)p, sizeof(T) * count);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        set_error("hipMalloc of %zu bytes failed: %s", sizeof(T) * count, hipGetErrorString(e));
        return LT_E_NOMEM;
    }
    return LT_OK;
}

template <typename T>
static void dfree(T *&p) {
    if (p) (void)hipFree((void *)p);
    p = nullptr;
}

// Room for n elements, whose old contents go.  cap is what p holds, also after a
// failure: a later job that needs less must not take the buffer for granted.
template <typename T>
static lt_status regrow(T **p, size_t &cap, size_t n) {
    if (cap >= n && *p) return LT_OK;
    dfree(*p);
    cap = 0;
    const lt_status s = dmalloc(p, n);
    if (s == LT_OK) cap = n;
    return s;
}

// Accumulates HIP-event intervals on one stream (GPUTimer, src/utils/Stopwatch.h:49-104).
struct EventTimer {
    std::vector<std::pair<hipEvent_t, hipEvent_t>> open;
    std::vector<hipEvent_t> pool;
    double ms = 0;
    uint64_t calls = 0;
    bool enabled = false;
    hipEvent_t take() {
        if (!pool.empty()) {
            hipEvent_t e = pool.back();
            pool.pop_back();
            return e;
        }
        hipEvent_t e;
        (void)hipEventCreate(&e);
        return e;
    }
    hipEvent_t begin(hipStream_t s) {
        calls++;
        if (!enabled) return nullptr;
        hipEvent_t a = take();
        (void)hipEventRecord(a, s);
        return a;
    }
    void end(hipEvent_t a, hipStream_t s) {
        if (!enabled || !a) return;
        hipEvent_t b = take();
        (void)hipEventRecord(b, s);
        open.emplace_back(a, b);
    }
    void collect() {
        for (auto &pr : open) {
            float t = 0;
            if (hipEventSynchronize(pr.second) == hipSuccess && hipEventElapsedTime(&t, pr.first, pr.second) == hipSuccess)
                ms += t;
            pool.push_back(pr.first);
            pool.push_back(pr.second);
        }
        open.clear();
    }
    void reset() {
        collect();
        ms = 0;
        calls = 0;
    }
    ~EventTimer() {
        collect();
        for (auto e : pool) (void)hipEventDestroy(e);
    }
};

// h_out: kNumStats u64 of event counters, the sequence number, those of the
// ring's buffers, that of the last load finished, then small results.
constexpr uint32_t kOutFlag = 2 * kNumStats, kOutRing = kOutFlag + 1, kOutCopy = 32, kOutData = 64;
constexpr uint64_t kManyOut = 1u << 20;  // words: from here on threads help with the results

struct RunSpec {
    int app = APP_PAGERANK;
    uint64_t total = 0;     // walker ids [0, total)
    uint32_t length = 0;    // pagerank / genericwalk l
    uint32_t source = 0;    // ppr
    float prob = 0.15f;     // ppr
    uint64_t nominal = 0;   // nominal steps for the stats
    // batched ppr
    const uint32_t *q_src = nullptr;
    const uint64_t *q_cnt = nullptr;
    uint32_t nq = 0;
    uint32_t *paths_out = nullptr;  // genericwalk: u32[total][length + 1] on the host
};

using WalkFn = void (*)(WalkArgs);
template <int APP>
static WalkFn walk_fn_app(int wpt, bool gen) {
    if (gen) return wpt == 4 ? walk_kernel<APP, 4, true> : wpt == 2 ? walk_kernel<APP, 2, true> : walk_kernel<APP, 1, true>;
    return wpt == 4 ? walk_kernel<APP, 4, false> : wpt == 2 ? walk_kernel<APP, 2, false> : walk_kernel<APP, 1, false>;
}
static WalkFn walk_fn(int app, int wpt, bool gen) {
    return app == APP_PAGERANK ? walk_fn_app<APP_PAGERANK>(wpt, gen)
           : app == APP_PPR    ? walk_fn_app<APP_PPR>(wpt, gen)
                               : walk_fn_app<APP_GENERIC>(wpt, gen);
}

struct Engine {
    const lt_graph *g = nullptr;
    lt_partition part;
    lt_config cfg;
    int device = 0;
    uint32_t V = 0, P = 0;
    hipStream_t s_compute = nullptr, s_copy = nullptr;
    int num_cu = 0;
    int max_grid = 0;           // init kernel (4 walkers per thread)
    int walk_grid[3][5] = {};  // resident workgroups of each walk kernel, by app and walkers per thread

    // partition table
    uint32_t *d_node_off = nullptr;
    uint64_t *d_edge_off = nullptr;
    uint32_t *d_lut = nullptr;
    uint32_t lut_shift = 0;
    PartRec *d_rec = nullptr;

    // HBM partition cache
    uint32_t nslots = 0;
    uint64_t slot_sz = 0;        // bytes per slot (256-aligned)
    bool slot_packed = false;    // slots keep columns packed (pack_partitions = 2)
    uint8_t *d_slots = nullptr;
    // One raw slot per partition: the slots are slices of one rowptr and one
    // col array (at most as many bytes), which run_flat walks directly.
    bool flat = false;
    lt_status alloc_flat();
    uint64_t *flat_rowptr = nullptr;   // [V+1], in d_slots
    uint32_t *flat_col = nullptr;      // [E], in d_slots
    uint32_t *d_rowptr32 = nullptr;    // [V+1] copy of flat_rowptr once every partition is cached (E < 2^32)
    bool rowptr32_set = false;         // it has been written
    std::vector<int32_t> slot_of;      // partition -> slot or -1
    std::vector<int32_t> part_in_slot; // slot -> partition or -1
    std::vector<uint32_t> free_slots;
    std::vector<uint8_t> resident;     // partition -> 0/1
    uint64_t zc_threshold = 0;
    const uint64_t *zc_rowptr = nullptr;  // device view of the pinned host graph
    const uint32_t *zc_col = nullptr;
    // Packed copies: images land in two HBM staging buffers by DMA on s_dma;
    // s_copy waits for the DMA, then unpacks into the slot, so the next DMA
    // overlaps this unpack.  Loads are complete when s_copy reaches them.
    // With too few hardware queues s_dma is s_copy (DMA and unpack in turn).
    std::shared_ptr<const PackedImage> pk_hold;  // packed partition images (pack_partitions)
    const PackedImage *pk = nullptr;
    uint8_t *d_stage[2] = {nullptr, nullptr};
    hipEvent_t stage_free[2] = {nullptr, nullptr};  // unpack of the buffer's last image done
    bool stage_used[2] = {false, false};
    uint32_t stage_next = 0;
    hipStream_t s_dma = nullptr;          // == s_copy without packed copies
    hipEvent_t ev_dma = nullptr;          // last DMA queued on s_dma

    // walker queues
    uint64_t wcap = 0;  // walkers the pool is sized for
    Queues q{};
    uint32_t *d_meta = nullptr;   // [P] qlen followed by PoolCtl
    uint64_t *h_packed = nullptr; // q.packed in pinned memory
    std::vector<uint32_t> h_meta; // what it last said: queue lengths, PoolCtl, the log's fill
    std::vector<uint64_t> counts; // walkers queued per partition: device queue + spilled to host
    std::vector<uint64_t> dcounts;  // device part of counts (qlen)

    // Host walker spill (src/WalkManager.h:11-58, src/Scheduler.h:53-82,
    // 215-233): with more walkers than num_device_walkers, whole device
    // queues move to per-partition queues in pinned, mapped host memory, and
    // come back when their partition is walked (the kernel reads them over
    // PCIe).  Host chunks are kChunk walkers, handed out from pinned blocks.
    static constexpr uint32_t kHostBlockChunks = 256;  // 16 MiB per pinned block
    bool spill_on = false;
    uint64_t dev_cap = 0;                   // walkers the device queues may hold
    std::vector<Walker *> hblocks, hblocks_dev;
    std::vector<uint32_t> hfree;            // free host chunk ids
    std::vector<std::deque<uint32_t>> hq;   // per partition: host chunks, oldest first
    std::vector<uint64_t> hhead, hcount;    // first walker's slot in hq[p].front(); walkers
    uint64_t spill_h2d_bytes = 0;           // spilled walkers read back over PCIe
    Walker *host_chunk_ptr(uint32_t id, bool dev) const {
        return (dev ? hblocks_dev : hblocks)[id / kHostBlockChunks] + (size_t)(id % kHostBlockChunks) * kChunk;
    }
    lt_status host_chunk(uint32_t &id);
    void host_reset();
    int32_t spill_victim(uint32_t except) const;
    lt_status spill_round(const std::vector<uint32_t> &victims);
    uint8_t *d_plan = nullptr, *h_plan = nullptr;  // spill round plan (device copy, pinned staging)
    size_t plan_cap = 0;
    lt_status ensure_room(uint64_t want, uint32_t except, uint64_t &room);
    lt_status process_host(uint32_t p, const WalkArgs &a);

    // outputs and statistics
    uint32_t *d_counts = nullptr;
    size_t counts_cap = 0;
    uint32_t count_copies = 1;  // 1 or kCountCopies arrays of V counts
    // Visit log of the running job (lt_visits.h) and the scratch it is counted with.
    uint32_t nbins = 0;
    VisitLog vl{};
    VisitScratch vs{};
    unsigned long long *d_vcur = nullptr;
    uint64_t vlog_cap = 0;                       // entries allocated
    uint64_t log_missed = 0;                     // visits counted directly for want of one
    uint32_t vregion = 0;                        // entries per region of the running job, 0 = no log
    bool wants_log(uint64_t visits, bool queued);
    bool ensure_log(uint64_t visits);
    void drop_log();
    lt_status count_log(uint32_t n, uint32_t most);
    uint32_t *d_endpoints = nullptr;
    size_t endpoints_cap = 0;
    uint32_t *d_moves = nullptr;
    uint32_t *d_paths = nullptr;
    size_t paths_cap = 0;
    size_t moves_cap = 0;
    uint64_t *d_qoff = nullptr;
    uint32_t *d_qsrc = nullptr;
    size_t qoff_cap = 0, qsrc_cap = 0;
    unsigned long long *d_stats = nullptr;
    // Results on their way to the caller (lt_results.h).
    static constexpr uint32_t kRing = 4;
    static constexpr size_t kRingBytes = 2u << 20, kRingSmall = 512u << 10;  // of a buffer
    uint32_t *h_out = nullptr, *d_out = nullptr;  // pinned: event counters, sequence number, small results
    uint32_t out_seq = 0;
    bool over = false;                            // the running job's walks were seen to be over,
    std::chrono::steady_clock::time_point t_over; // and when
    uint8_t *h_ring = nullptr, *d_ring = nullptr; // pinned: kRing buffers
    uint32_t ring_seq[kRing] = {};                // of each buffer's last fill
    std::vector<OutSeg> outs;                     // results of the running job
    uint8_t *h_query = nullptr;                   // pinned staging of the query table
    size_t query_cap = 0;
    lt_status poll_host(const uint32_t *flag, uint32_t seq, const char *what);
    lt_status finish_job(bool small);
    bool walks_over();
    lt_status wait_walks();
    static constexpr size_t kRingLarge = kRing * kRingBytes;
    size_t ring_cap = 0;       // bytes of the ring: 0, kRing * kRingSmall or kRingLarge
    size_t ring_seen = 0;      // of them, read by the CPU before
    uint64_t ring_words = 0;   // results for the large ring that went through the small one
    uint8_t *h_next = nullptr, *d_next = nullptr;  // the large ring until next_seen, what was read of it, is all
    size_t next_seen = 0;
    bool reading_next = false;  // the running job's helpers read it
    void start_results(ResultHelpers &help, bool cover);
    void swap_ring();
    lt_status mark_ring(uint32_t slot);
    lt_status wait_ring(uint32_t slot);
    lt_status copy_results(ResultHelpers &help);

    lt_stats st{};
    std::vector<lt_trace_rec> trace;
    std::vector<uint32_t> trace_counts;  // queue lengths seen by each traced decision
    std::vector<uint8_t> trace_resident; // residency seen by each traced decision
    std::vector<int32_t> trace_recent;   // last kRecent loads at each traced decision
    std::vector<uint32_t> trace_age;     // partition ages seen by each traced decision
    // Recency of HBM use, a scorer feature: use_clock counts the walks of
    // resident partitions since the engine was created, last_use[p] is the
    // clock after p's last one (0 = never), and p's age is their difference.
    std::vector<uint64_t> last_use;
    uint64_t use_clock = 0;
    Scorer *scorer = nullptr;             // learned policy (not owned)
    // device-side scheduling state (mirrors of slot_of / part_in_slot / resident)
    DevSched *d_ds = nullptr;
    int32_t *d_slot_of = nullptr, *d_part_in_slot = nullptr;
    uint8_t *d_resident = nullptr;
    bool rp_resident = false;      // rowptr of the whole graph kept in HBM (zc_rowptr points there)
    uint64_t *d_pk_off = nullptr, *d_pk_size = nullptr;  // device loop with block slots: image table
    const uint8_t *d_pk_img = nullptr;                     // device view of the pinned images (block slots)
    uint64_t *d_rowptr_all = nullptr;
    uint64_t pending_h2d = 0;      // one-off H2D bytes not yet charged to a run
    uint32_t zc_batch = 1;         // partitions per zero-copy launch
    uint32_t res_batch = 1;        // partitions per launch over resident queues
    uint32_t slice = kSliceChunks;
    std::vector<float> scores;            // scorer output of the current decision
    bool scores_valid = false;
    uint64_t scores_clock = 0;            // use_clock when the scores were computed
    bool infer_pending = false;           // an inference launched by infer_launch, not yet collected
    uint64_t pending_clock = 0;           // use_clock at its launch
    uint64_t w_run = 0;                   // walkers of the current wave
    EventTimer t_load, t_compute, t_zc, t_wload, t_wevict, t_kernel, t_kzc;  // t_kzc: walk launches over PCIe
    Scheduler sched;

    ~Engine();
    lt_status init(const lt_graph *g_, const lt_partition *p_, const lt_config *c);
    lt_status ensure_pool(uint64_t walkers, bool check_only = false);
    lt_status ensure_outputs(const RunSpec &rs, bool want_endpoints, bool want_moves);
    lt_status ensure_memory(const RunSpec &rs, uint64_t walkers, bool counting, bool want_endpoints, bool want_moves,
                            bool &walk_flat);
    lt_status run(const RunSpec &rs, uint32_t *counts_out, uint32_t *endpoints_out, uint32_t *moves_out);

    // scheduler primitives
    lt_status read_meta();
    // A load on its way.  Loads finish in order; h_out holds the number of the
    // last one that a kernel made.
    struct Load {
        bool pulled = false;     // by pull_kernel: seq is written when it is over
        uint32_t seq = 0;
        hipEvent_t ev = nullptr; // by DMA, with others behind it; else the copy stream itself is asked
    };
    uint32_t copy_seq = 0;
    std::vector<hipEvent_t> all_events, pool_events;  // of loads; those not in use
    uint32_t loading = 0;  // partitions that hold a slot and are not resident yet
    lt_status arrived(uint32_t p);
    lt_status drop_loads();
    bool loaded(const Load &l) const;
    lt_status wait_loaded(Load &l);
    bool meta_dirty = true;  // q.packed may be older than the queues
    uint32_t meta_seq = 0;   // of the last launch that writes q.packed
    bool meta_seen = true;   // h_meta holds what that launch wrote
    lt_status launch_fixup(Consumed d);
    lt_status wait_meta();
    TableBatch table_due{};  // table updates of the next walk launch
    TableFew table_told{};  // of the walk whose fix-up comes next
    lt_status flush_tables();
    lt_status process(uint32_t p, bool zerocopy, uint64_t walkers_hint);
    lt_status process_zc(uint32_t c, const uint8_t *pending);
    lt_status walk_batch(const std::vector<uint32_t> &parts, bool zerocopy);
    lt_status process_resident(uint32_t c, int kind, uint8_t *prefetched);
    void record(uint32_t p, int kind, int32_t loaded, int32_t evicted);
    lt_status evict(uint32_t p);
    lt_status load_async(uint32_t p, bool ahead, Load &l);
    lt_status copy_partition(uint32_t p, uint64_t *rp, uint32_t *cp);
    // Small slices are copied by one kernel instead of two DMAs, whose second
    // costs 10 us of its own (256 KB: 14 us, 22 by DMAs; 1 MB: 28 and 38).  Larger
    // ones hold the walks beside them up, which wait longer for memory.  In ms a job,
    // pulled and by DMAs: where walks go through all that is resident, s20 ppr 1 MB 14.5 and
    // 15.4, 1.25 MB 13.2 and 14.3, s21 pagerank 0.75 MB 10.2 and 11.0, 1.25 MB 6.2 and 6.1,
    // 1.5 MB 5.3 and 4.9; where a walk stays in one partition and a round has little
    // else to do, s18 pagerank 64 KB 58 and 61, 128 KB 58 and 61, 256 KB 32.2 and 31.9, s16
    // 6.7 and 6.9, s20 0.75 MB 55 and 50, 1 MB 40 and 35.
    static constexpr size_t kPullBytes = 1280u << 10, kPullBytesOne = 256u << 10;
    static constexpr int kPullGrid = 64;
    bool pulls(uint32_t p) const {
        const bool packed = pk && pk->size[p];
        if (packed && !slot_packed) return false;
        const size_t rbytes = ((size_t)part.node_off[p + 1] - part.node_off[p] + 1) * 8;
        return rbytes + (packed ? pk->size[p] : (part.edge_off[p + 1] - part.edge_off[p]) * 4) <=
               (cfg.span == LT_SPAN_RESIDENT ? kPullBytes : kPullBytesOne);
    }
    lt_status fetch_partition(uint32_t p, uint64_t *rowptr_out, uint32_t *col_out);
    // Bit streams of p's slot whose column part starts at cp: past the block
    // headers when the slot holds p's block image, nullptr for raw columns.
    const uint32_t *slot_words(uint32_t p, const uint32_t *cp) const {
        if (!slot_packed || !pk->size[p]) return nullptr;
        const uint64_t nblk = (part.edge_off[p + 1] - part.edge_off[p] + kBlockEdges - 1) / kBlockEdges;
        return cp + 2 * (nblk + 1);
    }
    // Where p's cached rowptr and col slices lie.
    void slot_ptrs(uint32_t p, uint64_t **rp, uint32_t **cp) const {
        if (flat) {
            *rp = flat_rowptr + part.node_off[p];
            *cp = flat_col + part.edge_off[p];
        } else {
            uint8_t *base = d_slots + (size_t)slot_of[p] * slot_sz;
            *rp = (uint64_t *)base;
            *cp = (uint32_t *)(base + ((uint64_t)part.node_off[p + 1] - part.node_off[p] + 1) * 8);
        }
    }
    lt_status set_table(uint32_t p, bool present);
    bool can_run_flat(const RunSpec &rs, uint32_t &missing) const;
    lt_status load_missing(ResultHelpers &help);
    lt_status run_flat(const RunSpec &rs, ResultHelpers &help);
    bool job_finished = false;  // run_flat has handed the job's results out
    lt_status scheduler_loop();
    lt_status scheduler_loop_learned();
    lt_status scheduler_loop_device();
    SchedState sched_state(bool device) const;
    lt_status infer_scores(int32_t cur);
    lt_status infer_launch(int32_t cur);
    lt_status infer_collect();
    int32_t learned_victim(int32_t a, int32_t b);
    void recent_loads(int32_t *out) const;
    uint32_t age_of(uint32_t p) const;
    // scores at most kStaleWalks walks of resident partitions old (the ages
    // and residency they saw have moved by at most that much)
    static constexpr uint64_t kStaleWalks = 16;
    bool scores_recent() const { return scores_valid && use_clock - scores_clock <= kStaleWalks; }
    lt_status run_partition(uint32_t p, int32_t &prev_loaded);

    AppArgs app{};
    int app_kind = APP_PAGERANK;
    size_t lds_bytes(int wpt = kWpt) const { return append_lds_bytes(P, wpt); }
    bool append_gen() const { return P > kDirectMaxP || cfg.append_mode != 0; }
    lt_status launch_walk(WalkArgs &a, uint64_t walkers, hipStream_t s);
    uint64_t partition_bytes(uint32_t p) const {
        return ((uint64_t)part.node_off[p + 1] - part.node_off[p] + 1) * 8 +
               (part.edge_off[p + 1] - part.edge_off[p]) * 4;
    }
};

Engine::~Engine() {
    if (s_compute) (void)hipStreamSynchronize(s_compute);
    if (s_copy) (void)hipStreamSynchronize(s_copy);
    if (s_dma && s_dma != s_copy) (void)hipStreamSynchronize(s_dma);
    for (auto ev : all_events) (void)hipEventDestroy(ev);
    dfree(d_node_off);
    dfree(d_edge_off);
    dfree(d_lut);
    dfree(d_rec);
    dfree(d_slots);
    dfree(d_rowptr32);
    dfree(q.slab);
    dfree(q.frame);
    dfree(q.free_stack);
    dfree(q.lost);
    dfree(d_meta);
    if (h_packed) (void)hipHostFree(h_packed);
    for (Walker *b : hblocks) (void)hipHostFree(b);
    dfree(d_plan);
    if (h_plan) (void)hipHostFree(h_plan);
    dfree(d_counts);
    dfree(vl.log);
    dfree(d_vcur);
    dfree(d_endpoints);
    dfree(d_moves);
    dfree(d_paths);
    dfree(d_qoff);
    dfree(d_qsrc);
    dfree(d_stats);
    if (h_out) (void)hipHostFree(h_out);
    if (h_ring) (void)hipHostFree(h_ring);
    if (h_next) (void)hipHostFree(h_next);
    if (h_query) (void)hipHostFree(h_query);
    dfree(d_ds);
    dfree(d_slot_of);
    dfree(d_part_in_slot);
    dfree(d_resident);
    dfree(d_rowptr_all);
    dfree(d_pk_off);
    dfree(d_pk_size);
    dfree(d_stage[0]);
    dfree(d_stage[1]);
    if (s_compute) (void)hipStreamDestroy(s_compute);
    if (s_copy) (void)hipStreamDestroy(s_copy);
    if (s_dma && s_dma != s_copy) (void)hipStreamDestroy(s_dma);
    for (int k = 0; k < 2; k++)
        if (stage_free[k]) (void)hipEventDestroy(stage_free[k]);
    if (ev_dma) (void)hipEventDestroy(ev_dma);
}

lt_status Engine::init(const lt_graph *g_, const lt_partition *p_, const lt_config *c) {
    g = g_;
    part = *p_;
    cfg = *c;
    V = g->V;
    P = part.P();
    LT_TRY(check_partition_of(*g, part));
    if (P > kMaxPartitions) {
        set_error("%u partitions exceed the engine limit %u; use a larger partition size", P, kMaxPartitions);
        return LT_E_ARG;
    }
    if (V == 0) {
        set_error("empty graph");
        return LT_E_ARG;
    }
    if (cfg.evict_shortlist < 0) {
        set_error("evict_shortlist must be >= 0 (got %d)", cfg.evict_shortlist);
        return LT_E_ARG;
    }
    if (cfg.append_mode < 0 || cfg.append_mode > 2) {
        set_error("append_mode must be 0, 1 or 2 (got %d)", cfg.append_mode);
        return LT_E_ARG;
    }
    if (cfg.learned_next < 0 || cfg.learned_next > 100) {
        set_error("learned_next must be 0-100 (got %d)", cfg.learned_next);
        return LT_E_ARG;
    }
    if (cfg.prefetch_plain < 0 || cfg.prefetch_plain > 2) {
        set_error("prefetch_plain must be 0, 1 or 2 (got %d)", cfg.prefetch_plain);
        return LT_E_ARG;
    }
    if (cfg.walkers_per_thread != 0 && cfg.walkers_per_thread != 1 && cfg.walkers_per_thread != 2 &&
        cfg.walkers_per_thread != 4) {
        set_error("walkers_per_thread must be 0, 1, 2 or 4 (got %d)", cfg.walkers_per_thread);
        return LT_E_ARG;
    }
    if (cfg.pack_partitions < 0 || cfg.pack_partitions > 2) {
        set_error("pack_partitions must be 0, 1 or 2 (got %d)", cfg.pack_partitions);
        return LT_E_ARG;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
        (void)hipGetLastError();
        set_error("no HIP device visible");
        return LT_E_NODEVICE;
    }
    if (!g->pinned) {
        set_error("graph was loaded without a HIP device; reopen it");
        return LT_E_ARG;
    }
    LT_HIP(hipSetDevice(device));
    hipDeviceProp_t prop;
    LT_HIP(hipGetDeviceProperties(&prop, device));
    num_cu = prop.multiProcessorCount;
    LT_HIP(hipStreamCreateWithFlags(&s_compute, hipStreamNonBlocking));
    LT_HIP(hipStreamCreateWithFlags(&s_copy, hipStreamNonBlocking));
    int occ = 0;
    LT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, init_kernel<APP_PAGERANK>, kBlock, lds_bytes()));
    max_grid = std::max(1, occ) * num_cu;
    // Each app's kernels have their own register counts, so their own
    // occupancy: a grid sized by another kernel's would queue workgroups
    // behind the resident ones and finish in a second, partial round.
    for (int app : {APP_PAGERANK, APP_PPR, APP_GENERIC})
        for (int wpt : {1, 2, 4}) {
            LT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void *)walk_fn(app, wpt, append_gen()),
                                                                kBlock, lds_bytes(wpt)));
            walk_grid[app][wpt] = std::max(1, occ) * num_cu;
        }

    // partition table + vertex -> partition lookup table
    LT_TRY(dmalloc(&d_node_off, P + 1));
    LT_TRY(dmalloc(&d_edge_off, P + 1));
    LT_HIP(hipMemcpy(d_node_off, part.node_off.data(), 4 * (P + 1), hipMemcpyHostToDevice));
    LT_HIP(hipMemcpy(d_edge_off, part.edge_off.data(), 8 * (P + 1), hipMemcpyHostToDevice));
    uint32_t bits = 0;
    while (bits < 32 && (1ull << bits) < (uint64_t)V) bits++;
    lut_shift = bits > 16 ? bits - 16 : 0;
    const size_t nlut = (((size_t)V - 1) >> lut_shift) + 1;
    std::vector<uint32_t> lut(nlut);
    for (size_t j = 0; j < nlut; j++) lut[j] = part.find((uint32_t)(j << lut_shift));
    LT_TRY(dmalloc(&d_lut, nlut));
    LT_HIP(hipMemcpy(d_lut, lut.data(), 4 * nlut, hipMemcpyHostToDevice));
    std::vector<PartRec> rec(P);
    for (uint32_t p = 0; p < P; p++)
        rec[p] = {nullptr, nullptr, nullptr, part.edge_off[p], part.node_off[p], part.node_off[p + 1]};
    LT_TRY(dmalloc(&d_rec, P));
    LT_HIP(hipMemcpy(d_rec, rec.data(), sizeof(PartRec) * P, hipMemcpyHostToDevice));

    // Packed copies: the images are built once per graph and partition table.
    // Format 1 travels gap-coded and is unpacked into raw slots; format 2 is
    // read in place, so slots are as large as the largest packed partition and
    // the same cache bytes hold more of them.
    s_dma = s_copy;
    // The device loop copies with load_kernel and has no unpack step: it
    // takes block slots (2), not gap-coded copies (1).
    if (cfg.pack_partitions == 2 || (cfg.pack_partitions == 1 && !cfg.device_schedule)) {
        LT_TRY(packed_image(*g, part, cfg.pack_partitions >= 2 ? 2 : 1, &pk_hold));
        pk = pk_hold.get();
        if (!pk->max_size) {
            pk = nullptr;  // no partition gets smaller
            pk_hold.reset();
        }
    }
    slot_packed = pk && pk->format == 2;
    // Blocks pay where they let more partitions stay. Asked for raw slots for all,
    // the images only travel, and the columns are kept raw, for flat walks: a
    // move reads one line of columns instead of two one after the other (s20
    // batched ppr, 5 M walkers: 4.05 ms a job from blocks, 1.65 so).  They take no more
    // than the slots asked for; not where they take more than a quarter of the
    // free memory, or cannot be allocated.
    if (slot_packed && !cfg.device_schedule && (cfg.num_device_partitions == 0 || cfg.num_device_partitions >= P)) {
        size_t room = 0, all = 0;
        LT_HIP(hipMemGetInfo(&room, &all));
        slot_packed = 8ull * ((uint64_t)V + 1) + 4ull * g->E > room / 4 || alloc_flat() != LT_OK;
    }

    // HBM cache slots (GPUGraph, src/GraphLoader.h:175-176)
    uint64_t slot_bytes = 0;
    slot_layout(part, slot_packed ? pk->size.data() : nullptr, cfg.num_device_partitions, &slot_bytes, &nslots);
    slot_sz = slot_bytes;
    // The whole rowptr array in HBM, paid for with slots of the same cache:
    // a zero-copied move then reads only its column entry over PCIe.
    const uint64_t rp_bytes = 8ull * ((uint64_t)V + 1);
    const uint32_t rp_slots = (uint32_t)((rp_bytes + slot_bytes - 1) / slot_bytes);
    // Off unless asked for: on R-MAT s26 pagerank with an 8 GB cache the
    // slots it takes cost about the PCIe bytes it saves at the default
    // threshold.  At least two slots stay, so that eviction, which spares the
    // partition loaded last, has a victim.
    rp_resident = cfg.rowptr_resident > 0;
    if (nslots == P) rp_resident = false;  // nothing is zero-copied with every partition cached
    if (rp_resident && nslots >= rp_slots + 2) nslots -= rp_slots;
    else rp_resident = false;
    flat = nslots == P && !slot_packed && !cfg.device_schedule;
    if (!flat) LT_TRY(dmalloc(&d_slots, (size_t)nslots * slot_bytes));
    else if (!d_slots) LT_TRY(alloc_flat());
    slot_of.assign(P, -1);
    part_in_slot.assign(nslots, -1);
    resident.assign(P, 0);
    last_use.assign(P, 0);
    free_slots.clear();
    for (uint32_t s = 0; s < nslots; s++) free_slots.push_back(nslots - 1 - s);
    // Default threshold: the reference's partitionSize / cachelineSize / 2
    // (src/Scheduler.h:295) for the plain policies.  The learned policy uses
    // the byte break-even instead: a zero-copied walker step reads a rowptr
    // pair and a column id, two 64-byte PCIe reads, so reading S bytes by DMA
    // costs the same as S/128 zero-copied walkers.
    if (cfg.zerocopy_threshold != UINT64_MAX) zc_threshold = cfg.zerocopy_threshold;
    else zc_threshold = cfg.policy == LT_SCHED_LEARNED ? part.bytes / 128 : part.bytes / 128 / 2;
    LT_HIP(hipHostGetDevicePointer((void **)&zc_rowptr, g->rowptr, 0));
    LT_HIP(hipHostGetDevicePointer((void **)&zc_col, g->col, 0));
    if (pk && !slot_packed) {  // staging buffers for the images unpacked in HBM
        for (int k = 0; k < 2; k++) {
            LT_TRY(dmalloc(&d_stage[k], pk->max_size));
            LT_HIP(hipEventCreateWithFlags(&stage_free[k], hipEventDisableTiming));
        }
        // HIP spreads streams over GPU_MAX_HW_QUEUES hardware queues (4
        // unless set).  A DMA stream that shares a queue with the walk
        // stream waits behind walk kernels, so it is used only when the
        // streams in play (null, walk, copy, DMA, a scorer's) get their own.
        const char *hwq = getenv("GPU_MAX_HW_QUEUES");
        if (hwq && atoi(hwq) >= 6) {
            LT_HIP(hipEventCreateWithFlags(&ev_dma, hipEventDisableTiming));
            LT_HIP(hipStreamCreateWithFlags(&s_dma, hipStreamNonBlocking));
        }
    }
    if (cfg.device_schedule && slot_packed) {  // the device loop's copies read the images in place
        std::vector<uint64_t> off(P), size(P);
        for (uint32_t i = 0; i < P; i++) {
            off[i] = pk->off[i];
            size[i] = pk->size[i];
        }
        LT_TRY(dmalloc(&d_pk_off, P));
        LT_TRY(dmalloc(&d_pk_size, P));
        LT_HIP(hipMemcpy(d_pk_off, off.data(), 8 * (size_t)P, hipMemcpyHostToDevice));
        LT_HIP(hipMemcpy(d_pk_size, size.data(), 8 * (size_t)P, hipMemcpyHostToDevice));
    }
    if (slot_packed) LT_HIP(hipHostGetDevicePointer((void **)&d_pk_img, pk->host, 0));
    if (rp_resident) {
        LT_TRY(dmalloc(&d_rowptr_all, (size_t)V + 1));
        LT_HIP(hipMemcpy(d_rowptr_all, g->rowptr, rp_bytes, hipMemcpyHostToDevice));
        pending_h2d = rp_bytes;  // charged to the first run
        zc_rowptr = d_rowptr_all;
    }

    // queue lengths one 128-byte line apart, then PoolCtl on its own line; the
    // fix-up kernel packs both into h_packed (pinned, mapped) for the host
    LT_TRY(dmalloc(&d_meta, (size_t)P * kQStride + kQStride));
    h_meta.assign(P + 4 + kLogRegions, 0);
    LT_HIP(hipHostMalloc((void **)&h_packed, 8 * h_meta.size(), hipHostMallocMapped | hipHostMallocCoherent));
    memset(h_packed, 0, 8 * h_meta.size());
    LT_HIP(hipHostGetDevicePointer((void **)&q.packed, h_packed, 0));
    q.qlen = d_meta;
    q.ctl = (PoolCtl *)(d_meta + (size_t)P * kQStride);
    q.P = P;
    nbins = (uint32_t)(((uint64_t)V + kBin - 1) / kBin);
    if (cfg.device_schedule) {
        LT_TRY(dmalloc(&d_ds, 1));
        LT_TRY(dmalloc(&d_slot_of, P));
        LT_TRY(dmalloc(&d_part_in_slot, nslots));
        LT_TRY(dmalloc(&d_resident, P));
    }
    zc_batch = cfg.zc_batch > 0 ? (uint32_t)cfg.zc_batch
                                : (cfg.policy == LT_SCHED_LEARNED && cfg.span == LT_SPAN_RESIDENT ? kMaxZcBatch : 1);
    zc_batch = std::min(zc_batch, kMaxZcBatch);
    if (cfg.span != LT_SPAN_RESIDENT) zc_batch = 1;  // a batch relies on walking through the table
    res_batch = cfg.resident_batch > 0
                    ? (uint32_t)cfg.resident_batch
                    : (cfg.policy == LT_SCHED_LEARNED && cfg.span == LT_SPAN_RESIDENT ? kMaxZcBatch : 1);
    res_batch = std::min(res_batch, kMaxZcBatch);
    if (cfg.span != LT_SPAN_RESIDENT) res_batch = 1;
    slice = cfg.slice_chunks > 0 ? (uint32_t)cfg.slice_chunks : kSliceChunks;
    LT_TRY(dmalloc(&d_stats, (size_t)kNumStats * kStatSlots));
    LT_HIP(hipHostMalloc((void **)&h_out, 4 * (kOutData + kSmallOut), hipHostMallocMapped | hipHostMallocCoherent));
    memset(h_out, 0, 4 * kOutData);
    LT_HIP(hipHostGetDevicePointer((void **)&d_out, h_out, 0));
    counts.assign(P, 0);
    dcounts.assign(P, 0);
    hq.assign(P, {});
    hhead.assign(P, 0);
    hcount.assign(P, 0);

    bool timers = cfg.event_timers != 0;
    t_load.enabled = t_compute.enabled = t_zc.enabled = t_wload.enabled = t_wevict.enabled = timers;
    t_kernel.enabled = t_kzc.enabled = timers;
    sched.init(P, cfg);
    return LT_OK;
}

// The slots of a flat cache.
lt_status Engine::alloc_flat() {
    const size_t rp_size = (8 * ((size_t)V + 1) + 255) & ~(size_t)255;
    LT_TRY(dmalloc(&d_slots, rp_size + 4 * (size_t)g->E));
    flat_rowptr = (uint64_t *)d_slots;
    flat_col = (uint32_t *)(d_slots + rp_size);
    return LT_OK;
}

// Size the chunk pool for `walkers` queued walkers: every queue may hold a
// partly filled chunk, the slice being consumed keeps its chunks until the
// fix-up, and allocation races may strand up to kLostCap chunks per launch.
// check_only: refuse what the queues could not hold, allocate nothing.
lt_status Engine::ensure_pool(uint64_t walkers, bool check_only) {
    if (walkers <= wcap && q.slab) return LT_OK;
    const uint64_t wchunks = (walkers + kChunk - 1) / kChunk;
    // one launch holds at most `held` source chunks while filling new ones
    const uint64_t held = cfg.device_schedule ? wchunks + 1 : std::min<uint64_t>(slice, wchunks + 1);
    // A reservation links at most two chunks and so loses at most two, and a launch
    // makes one for each pass and partition (a pass has kBlock walkers or more; 128: queues
    // and pieces that end in a short one).  With few partitions that is far below
    // kLostCap: 46 MB instead of 268 for 90 000 walkers of one, whose allocation took
    // a new engine's first job half its time.
    const uint64_t lost = cfg.append_mode == 2 ? kLostCap
                                               : std::min<uint64_t>(kLostCap, 2 * (uint64_t)P * (walkers / kBlock + 128));
    const uint64_t nchunks = wchunks + P + held + 2 + lost;
    const uint64_t maxc = wchunks + 2;
    if (nchunks >= 0xFFFFFFF0ull || maxc * kChunk > 0xFFFFFFFFull) {
        set_error("%llu walkers exceed the queue limits; lower -b", (unsigned long long)walkers);
        return LT_E_ARG;
    }
    if (check_only) return LT_OK;
    wcap = 0;  // until all four are there
    dfree(q.slab);
    dfree(q.frame);
    dfree(q.free_stack);
    dfree(q.lost);
    q.nchunks = (uint32_t)nchunks;
    q.maxc = (uint32_t)maxc;
    LT_TRY(dmalloc(&q.slab, (size_t)nchunks * kChunk));
    LT_TRY(dmalloc(&q.frame, (size_t)P * maxc));
    LT_TRY(dmalloc(&q.free_stack, nchunks));
    LT_TRY(dmalloc(&q.lost, kLostCap));
    wcap = walkers;
    return LT_OK;
}

lt_status Engine::ensure_outputs(const RunSpec &rs, bool want_endpoints, bool want_moves) {
    LT_TRY(regrow(&d_counts, counts_cap, (size_t)V * count_copies));
    if (want_endpoints) LT_TRY(regrow(&d_endpoints, endpoints_cap, rs.total));
    if (rs.paths_out) LT_TRY(regrow(&d_paths, paths_cap, (size_t)rs.total * ((size_t)rs.length + 1)));
    if (want_moves) LT_TRY(regrow(&d_moves, moves_cap, rs.total));
    if (rs.nq) {
        LT_TRY(regrow(&d_qoff, qoff_cap, (size_t)rs.nq + 1));
        LT_TRY(regrow(&d_qsrc, qsrc_cap, rs.nq));
    }
    return LT_OK;
}

// Log for a job of `visits` visits, or none (vregion = 0).  A flat job has one from
// kLogVisits on: below, the counters' atomics (27 G/s) cost less than the
// launches that count a log, 10 to 30 us.  A job that goes through the queues walks
// a few thousand visits a launch when it is small, and their atomics overlap
// its other waits: 14 M visits in 900 launches took 33.0 ms directly and 35.0 with
// a log, 103 M in 72 launches 18.4 and 15.1.  Above kMaxBins bins (67 M
// vertices) the scatter's LDS does not hold a tile's histogram, and a device
// that cannot hold a log counts directly.
constexpr uint64_t kLogVisits = 1u << 18, kLogVisitsQueued = 1u << 24;
constexpr uint64_t kLogMost = 1ull << 26;  // entries: 256 MB; 0.75 GB with what counting them takes
// A flat job allocates a log once that many visits were counted without: their
// atomics have then cost what the allocation takes, 13 to 20 us a million visits
// and 50 to 600 us.  (Allocated by any engine's second job, it took that one
// from 90 to 600 us on s16, 0.9 M visits a job, and from 54 to 600 on s14, 0.3 M.)
constexpr uint64_t kLogPays = 1ull << 25;

// Entries of a job's log: regions fill unevenly, so a quarter more than its visits,
// and a launch's workgroups' buffers.
static uint64_t log_entries(uint64_t visits) {
    visits = std::min(visits, kLogMost);
    return std::min(kLogMost, visits + visits / 4 + (1u << 20)) & ~(uint64_t)(kTile * kLogRegions - 1);
}

bool Engine::wants_log(uint64_t visits, bool queued) {
    if (visits < (queued ? kLogVisitsQueued : kLogVisits) || nbins > kMaxBins) return false;
    if (queued || vlog_cap >= log_entries(visits)) return true;
    log_missed += std::min(visits, kLogPays);
    if (log_missed < kLogPays) return false;
    log_missed = 0;
    return true;
}

// Whether there is memory for it.
bool Engine::ensure_log(uint64_t visits) {
    const uint64_t want = log_entries(visits);
    if (vlog_cap < want) {
        drop_log();
        const size_t cur = (size_t)kLogRegions * kCurStride;  // cursors, then the bins' totals and first units
        // The log and what counting a full one takes, in one allocation: one by
        // one they took a new engine's first job 0.6 ms, with tens of MB or few.
        const uint64_t tiles = want / kTile + kLogRegions;
        const uint64_t units = std::max<uint64_t>(nbins <= kFewBins ? std::min<uint64_t>(kFewUnits, tiles * nbins) : 0,
                                                  std::min<uint64_t>(want / kHistUnit, kHistUnits) + 1 + nbins);
        const uint64_t words[4] = {want, want / 2, tiles * nbins, units * kBin};  // multiples of 4 but the third
        if (dmalloc(&d_vcur, cur + nbins + 1) != LT_OK ||
            dmalloc(&vl.log, words[0] + words[1] + words[2] + 4 + words[3]) != LT_OK) {
            drop_log();
            return false;
        }
        vs.total = (uint32_t *)(d_vcur + cur);
        vs.unit_off = vs.total + nbins;
        vs.sorted = (uint16_t *)(vl.log + words[0]);
        vs.run = vl.log + words[0] + words[1];
        vs.partial = vs.run + ((words[2] + 3) & ~3ull);
        vlog_cap = want;
    }
    vregion = (uint32_t)(want / kLogRegions);
    return true;
}

void Engine::drop_log() {
    dfree(d_vcur);
    dfree(vl.log);
    vlog_cap = 0;
}

// Device memory of a job.  What it cannot do without comes first; the visit log, the
// counters' copies and the flat walks' row offsets give way to that, and none of
// these fails a job that does without.
lt_status Engine::ensure_memory(const RunSpec &rs, uint64_t walkers, bool counting, bool want_endpoints,
                                bool want_moves, bool &walk_flat) {
    uint64_t visits = rs.total;
    if (rs.app == APP_PAGERANK && __builtin_mul_overflow(rs.total, (uint64_t)rs.length, &visits)) visits = UINT64_MAX;
    vregion = 0;
    if (walk_flat && !d_rowptr32 && dmalloc(&d_rowptr32, (size_t)V + 1) != LT_OK) walk_flat = false;
    bool one = false;  // no copies
    bool log = counting && wants_log(visits, !walk_flat);
    while (true) {
        // Without a log, copies of the counters, one per XCD: where the walkers of
        // one launch stay in a few partitions (capped cache, PPR around its sources; one
        // array measured 29 % slower there), and where clearing and adding up the
        // copies of a small graph costs less than its hot vertices' atomics (5 G/s in
        // one array, 27 G/s in copies).
        const bool copies =
            (!walk_flat && (nslots < P || rs.app == APP_PPR)) || (visits >= (1u << 16) && V <= (1u << 20));
        count_copies = counting && !log && copies && !one ? kCountCopies : 1;
        lt_status s = ensure_pool(walkers, walk_flat);  // a flat job keeps the queues' limits
        if (s == LT_OK) s = ensure_outputs(rs, want_endpoints, want_moves);
        if (s == LT_OK) {
            if (!log || ensure_log(visits)) return LT_OK;
            log = false;
        } else if (s != LT_E_NOMEM) {
            return s;
        } else if (vl.log) {
            drop_log();
        } else if (count_copies > 1) {
            one = true;
        } else if (d_rowptr32) {
            dfree(d_rowptr32);
            rowptr32_set = walk_flat = false;
            log = log && wants_log(visits, true);
        } else {
            return s;
        }
    }
}

// Counts the log into d_counts and empties it: the n entries of a flat job's
// log, or (n = 0) the regions, which hold at most `most` entries each.
lt_status Engine::count_log(uint32_t n, uint32_t most) {
    VisitLog l = vl;
    l.cur = d_vcur;
    l.cap = n ? 0 : vregion;
    l.n = n;
    const uint64_t entries = n ? n : (uint64_t)std::min(most, vregion) * kLogRegions;
    if (entries == 0) return LT_OK;
    l.tiles = (uint32_t)(((n ? n : entries / kLogRegions) + kTile - 1) / kTile);
    const uint32_t ntiles = n ? l.tiles : l.tiles * kLogRegions;
    const bool few = nbins <= kFewBins && ntiles * nbins <= kFewUnits;
    vs.unit = std::max<uint32_t>(kHistUnit, (uint32_t)(entries / kHistUnits));
    const uint32_t units = few ? ntiles * nbins : (uint32_t)((entries + vs.unit - 1) / vs.unit) + nbins;
    if (few) {
        visit_hist_kernel<false><<<units, kVisitThreads, 0, s_compute>>>(l, vs, nbins, ntiles);
    } else {
        visit_tile_kernel<<<ntiles, kVisitThreads, 4 * kRepl * nbins, s_compute>>>(l, vs, nbins, ntiles);
        visit_scan_kernel<<<nbins, kVisitThreads, 0, s_compute>>>(vs, ntiles);
        visit_scatter_kernel<<<ntiles, kVisitThreads, scatter_lds(nbins), s_compute>>>(l, vs, nbins, ntiles);
        visit_hist_kernel<true><<<units, kVisitThreads, 0, s_compute>>>(l, vs, nbins, ntiles);
    }
    visit_sum_kernel<<<(V + 255) / 256, 256, 0, s_compute>>>(l, vs, d_counts, V);
    LT_HIP(hipGetLastError());
    return LT_OK;
}

lt_status Engine::launch_fixup(Consumed d) {
    q.seq = ++meta_seq;
    d.due = table_told;
    table_told.n = 0;
    fixup_kernel<<<1, kBlock, 0, s_compute>>>(q, d, d_rec);
    LT_HIP(hipGetLastError());
    meta_dirty = false;
    meta_seen = false;
    return LT_OK;
}

// Waits until every word of h_packed is of the last launch that writes it, and
// so until the walk before that launch is over.  Every decision waits here; the host
// polls the words' numbers: launch, fix-up and wait of a small kernel take
// 10 us so, 27 us when hipStreamQuery is polled and 12 us with
// hipStreamSynchronize.  A stream that ends or fails without a word being
// written is found by the query made once in a while.
lt_status Engine::wait_meta() {
    if (meta_seen) return LT_OK;
    const size_t n = P + 4 + (q.vcur ? kLogRegions : 0);
    for (size_t i = 0; i < n; i++) {
        LT_TRY(poll_host((const uint32_t *)(h_packed + i) + 1, meta_seq, "queue lengths"));
        h_meta[i] = (uint32_t)h_packed[i];
    }
    meta_seen = true;
    return LT_OK;
}

lt_status Engine::poll_host(const uint32_t *flag, uint32_t seq, const char *what) {
    for (uint32_t it = 1; __atomic_load_n(flag, __ATOMIC_ACQUIRE) != seq; it++) {
        __builtin_ia32_pause();
        if ((it & 0xFFFFF) == 0) {
            const hipError_t e = hipStreamQuery(s_compute);
            if (e == hipErrorNotReady) continue;
            LT_HIP(e);
            if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq) break;
            set_error("%s were not written", what);
            return LT_E_INTERNAL;
        }
    }
    return LT_OK;
}

lt_status Engine::read_meta() {
    if (meta_dirty) {  // the last queue update on s_compute was not followed by a fix-up
        q.seq = ++meta_seq;
        pack_meta_kernel<<<1, kBlock, 0, s_compute>>>(q);
        LT_HIP(hipGetLastError());
        meta_dirty = false;
        meta_seen = false;
    }
    LT_TRY(wait_meta());
    const PoolCtl *c = (const PoolCtl *)&h_meta[P];
    if (c->overflow) {
        set_error("walker queue pool overflow (flags 0x%x, top %u)", c->overflow, c->top);
        return LT_E_INTERNAL;
    }
    for (uint32_t i = 0; i < P; i++) {
        dcounts[i] = h_meta[i];
        counts[i] = dcounts[i] + hcount[i];
    }
    if (vregion) {  // the log is counted before its fullest region is full
        const uint32_t *cur = &h_meta[P + 4];
        const uint32_t most = *std::max_element(cur, cur + kLogRegions);
        if (most >= vregion / 5 * 4) {
            LT_TRY(count_log(0, most));
            meta_dirty = true;
            for (uint32_t r = 0; r < kLogRegions; r++) h_meta[P + 4 + r] = 0;
        }
    }
    return LT_OK;
}

// Queue a table update for the next walk launch that reads tables (flush_tables).
lt_status Engine::set_table(uint32_t p, bool present) {
    uint32_t k = 0;
    while (k < table_due.n && table_due.part[k] != p) k++;  // the last update of a partition counts
    if (k == kTableBatch) {
        LT_TRY(flush_tables());
        k = 0;
    }
    if (k == table_due.n) table_due.n++;
    table_due.part[k] = p;
    table_due.rowptr[k] = nullptr;
    table_due.col[k] = table_due.words[k] = nullptr;
    if (present) {
        uint64_t *r;
        uint32_t *c;
        slot_ptrs(p, &r, &c);
        table_due.rowptr[k] = r;
        table_due.col[k] = c;
        table_due.words[k] = slot_words(p, c);
    }
    return LT_OK;
}

lt_status Engine::flush_tables() {
    if (table_due.n == 0) return LT_OK;
    set_tables_kernel<<<1, 64, 0, s_compute>>>(d_rec, table_due);
    LT_HIP(hipGetLastError());
    table_due.n = 0;
    return LT_OK;
}

lt_status Engine::evict(uint32_t p) {
    const int32_t s = slot_of[p];
    if (s < 0) return LT_OK;
    LT_TRY(set_table(p, false));
    slot_of[p] = -1;
    part_in_slot[s] = -1;
    resident[p] = 0;
    free_slots.push_back((uint32_t)s);
    return LT_OK;
}

bool Engine::loaded(const Load &l) const {
    if (l.pulled) return (int32_t)(__atomic_load_n(h_out + kOutCopy, __ATOMIC_ACQUIRE) - l.seq) >= 0;
    return (l.ev ? hipEventQuery(l.ev) : hipStreamQuery(s_copy)) != hipErrorNotReady;
}

// A pulled load's number and an event are polled; the end of a DMA with nothing
// behind it is waited for by the runtime.
lt_status Engine::wait_loaded(Load &l) {
    if (!l.pulled && !l.ev) {
        LT_HIP(hipStreamSynchronize(s_copy));
        return LT_OK;
    }
    for (uint32_t it = 1; !loaded(l); it++) {
        __builtin_ia32_pause();
        if (l.pulled && (it & 0xFFFFF) == 0) {
            const hipError_t e = hipStreamQuery(s_copy);
            if (e == hipErrorNotReady) continue;
            LT_HIP(e);
            if (loaded(l)) break;
            set_error("a partition copy did not finish");
            return LT_E_INTERNAL;
        }
    }
    if (!l.ev) return LT_OK;
    const hipError_t e = hipEventQuery(l.ev);
    pool_events.push_back(l.ev);
    l.ev = nullptr;
    LT_HIP(e);
    return LT_OK;
}

// p's copy is complete: walks may read its slot.
lt_status Engine::arrived(uint32_t p) {
    resident[p] = 1;
    loading--;
    return set_table(p, true);
}

// Takes the slots of loads back that a job which ended with an error did not wait for.
lt_status Engine::drop_loads() {
    if (loading == 0) return LT_OK;
    LT_HIP(hipStreamSynchronize(s_copy));
    if (s_dma != s_copy) LT_HIP(hipStreamSynchronize(s_dma));
    for (uint32_t p = 0; p < P; p++) {
        if (slot_of[p] < 0 || resident[p]) continue;
        part_in_slot[slot_of[p]] = -1;
        free_slots.push_back((uint32_t)slot_of[p]);
        slot_of[p] = -1;
    }
    pool_events = all_events;
    loading = 0;
    return LT_OK;
}

// GPUGraph::loadAsync (src/GraphLoader.h:193-215): rowptr slice at slot offset
// 0, col slice right after it, both on the copy stream.  The compute stream
// must not be reading the slot (the caller evicted it after a sync).  ahead: other
// loads may follow before this one is waited for.
lt_status Engine::load_async(uint32_t p, bool ahead, Load &l) {
    if (free_slots.empty()) {
        set_error("no free cache slot for partition %u", p);
        return LT_E_INTERNAL;
    }
    const uint32_t s = free_slots.back();
    free_slots.pop_back();
    hipEvent_t t = t_load.begin(s_dma);
    slot_of[p] = (int32_t)s;
    part_in_slot[s] = (int32_t)p;
    loading++;
    uint64_t *rp;
    uint32_t *cp;
    slot_ptrs(p, &rp, &cp);
    LT_TRY(copy_partition(p, rp, cp));
    l = Load{};
    l.pulled = pulls(p);
    if (l.pulled) {  // (behind a DMA such a kernel starts 10 us late)
        l.seq = ++copy_seq;
        mark_kernel<<<1, 1, 0, s_copy>>>(d_out + kOutCopy, l.seq);
        LT_HIP(hipGetLastError());
    } else if (ahead) {
        if (pool_events.empty()) {
            LT_HIP(hipEventCreateWithFlags(&l.ev, hipEventDisableTiming));
            all_events.push_back(l.ev);
        } else {
            l.ev = pool_events.back();
            pool_events.pop_back();
        }
        LT_HIP(hipEventRecord(l.ev, s_copy));
    }
    t_load.end(t, s_copy);
    return LT_OK;
}

// Slot bytes of partition p: the rowptr slice at rp and the col slice at cp, either
// copied as is, or copied gap-coded into a staging buffer and unpacked from
// there, or (block slots) its block image copied into the slot, where it stays.
// The DMAs run on s_dma; s_copy waits for them (and unpacks), so the load is
// complete when s_copy reaches this point.  A staging buffer is refilled only
// after the unpack of its previous image.  Block slots copy on s_copy alone.
lt_status Engine::copy_partition(uint32_t p, uint64_t *rp, uint32_t *cp) {
    const uint32_t nb = part.node_off[p], ne = part.node_off[p + 1];
    const uint64_t eb = part.edge_off[p], ee = part.edge_off[p + 1];
    const size_t rbytes = ((size_t)ne - nb + 1) * 8, cbytes = (size_t)(ee - eb) * 4;
    const bool packed = pk && pk->size[p];
    uint32_t k = 0;
    if (pulls(p)) {
        const size_t body = packed ? pk->size[p] : cbytes;
        PullArgs a{};
        const uint32_t *col = zc_col + eb;
        if (packed) col = (const uint32_t *)(d_pk_img + pk->off[p]);
        a.src[0] = (const uint32_t *)(zc_rowptr + nb);
        a.src[1] = col;
        a.dst[0] = (uint32_t *)rp;
        a.dst[1] = cp;
        a.words[0] = rbytes / 4;
        a.words[1] = body / 4;
        pull_kernel<<<kPullGrid, 256, 0, s_copy>>>(a);
        LT_HIP(hipGetLastError());
        st.h2d_bytes_explicit += body + (rp_resident ? 0 : rbytes);
        st.h2d_bytes_unpacked += cbytes + (rp_resident ? 0 : rbytes);
        if (packed) {
            st.packed_image_bytes += body;
            st.packed_col_bytes += cbytes;
        }
        return LT_OK;
    }
    if (packed && slot_packed) {  // the block image is the slot's column part
        if (rp_resident) {
            LT_HIP(hipMemcpyAsync(rp, d_rowptr_all + nb, rbytes, hipMemcpyDeviceToDevice, s_copy));
        } else {
            LT_HIP(hipMemcpyAsync(rp, g->rowptr + nb, rbytes, hipMemcpyHostToDevice, s_copy));
            st.h2d_bytes_explicit += rbytes;
            st.h2d_bytes_unpacked += rbytes;
        }
        LT_HIP(hipMemcpyAsync(cp, pk->host + pk->off[p], pk->size[p], hipMemcpyHostToDevice, s_copy));
        st.h2d_bytes_unpacked += cbytes;
        st.h2d_bytes_explicit += pk->size[p];
        st.packed_image_bytes += pk->size[p];
        st.packed_col_bytes += cbytes;
        return LT_OK;
    }
    if (packed) {
        k = stage_next;
        stage_next ^= 1u;
        if (stage_used[k] && s_dma != s_copy) LT_HIP(hipStreamWaitEvent(s_dma, stage_free[k], 0));
    }
    if (rp_resident) {
        LT_HIP(hipMemcpyAsync(rp, d_rowptr_all + nb, rbytes, hipMemcpyDeviceToDevice, s_dma));
    } else {
        LT_HIP(hipMemcpyAsync(rp, g->rowptr + nb, rbytes, hipMemcpyHostToDevice, s_dma));
        st.h2d_bytes_explicit += rbytes;
        st.h2d_bytes_unpacked += rbytes;
    }
    st.h2d_bytes_unpacked += cbytes;
    if (packed) {
        LT_HIP(hipMemcpyAsync(d_stage[k], pk->host + pk->off[p], pk->size[p], hipMemcpyHostToDevice, s_dma));
        if (s_dma != s_copy) {
            LT_HIP(hipEventRecord(ev_dma, s_dma));
            LT_HIP(hipStreamWaitEvent(s_copy, ev_dma, 0));
        }
        if (pk->format == 2) {
            const int grid = (int)std::min<uint64_t>(8 * (uint64_t)num_cu, (ee - eb) / 256 + 1);
            unblock_kernel<<<grid, 256, 0, s_copy>>>((const uint32_t *)d_stage[k], ee - eb, cp);
        } else {
            const uint64_t n = ne - nb, nch = (ee - eb + 63) / 64;
            const uint64_t nwords = (pk->size[p] - 8 * nch) / 4 - 2;
            const uint64_t waves = (nch + kUnpackChunks - 1) / kUnpackChunks;
            unpack_kernel<<<(unsigned)((waves + 3) / 4), 256, 0, s_copy>>>(
                d_stage[k], (uint32_t)n, ee - eb, nwords, pk->vbits, rp, cp);
        }
        LT_HIP(hipGetLastError());
        LT_HIP(hipEventRecord(stage_free[k], s_copy));
        stage_used[k] = true;
        st.h2d_bytes_explicit += pk->size[p];
        st.packed_image_bytes += pk->size[p];
        st.packed_col_bytes += cbytes;
    } else {
        if (cbytes) LT_HIP(hipMemcpyAsync(cp, g->col + eb, cbytes, hipMemcpyHostToDevice, s_dma));
        st.h2d_bytes_explicit += cbytes;
        if (s_dma != s_copy) {
            LT_HIP(hipEventRecord(ev_dma, s_dma));
            LT_HIP(hipStreamWaitEvent(s_copy, ev_dma, 0));
        }
    }
    return LT_OK;
}

// A partition's slot bytes, built by copy_partition in a scratch buffer and
// copied back; the cache and the statistics are left as they were.
lt_status Engine::fetch_partition(uint32_t p, uint64_t *rowptr_out, uint32_t *col_out) {
    if (pk && pk->format == 2) {
        set_error("fetch of partition %u: refused with pack_partitions = 2, whose copies are block images", p);
        return LT_E_ARG;
    }
    LT_HIP(hipSetDevice(device));
    LT_HIP(hipStreamSynchronize(s_copy));
    if (s_dma != s_copy) LT_HIP(hipStreamSynchronize(s_dma));
    const size_t rn = (size_t)part.node_off[p + 1] - part.node_off[p] + 1;
    const size_t m = part.edge_off[p + 1] - part.edge_off[p];
    uint8_t *buf = nullptr;
    LT_TRY(dmalloc(&buf, rn * 8 + m * 4));
    const lt_stats keep = st;
    lt_status rc = copy_partition(p, (uint64_t *)buf, (uint32_t *)(buf + rn * 8));
    st = keep;
    hipError_t e = rc == LT_OK ? hipStreamSynchronize(s_copy) : hipSuccess;
    if (rc == LT_OK && e == hipSuccess) e = hipMemcpy(rowptr_out, buf, rn * 8, hipMemcpyDeviceToHost);
    if (rc == LT_OK && e == hipSuccess && m) e = hipMemcpy(col_out, buf + rn * 8, m * 4, hipMemcpyDeviceToHost);
    dfree(buf);
    if (rc != LT_OK) return rc;
    if (e != hipSuccess) {
        set_error("fetch of partition %u: %s", p, hipGetErrorString(e));
        return LT_E_HIP;
    }
    return LT_OK;
}

// Walk launch sized to the slice: 1 walker per thread while the slice is
// small enough that more walkers per thread would leave SIMDs without waves
// (a thread walks its walkers one after another), 2 or 4 for large slices,
// where the per-workgroup append cost (histogram, scan, one atomic per
// destination queue) is spread over more walkers.
lt_status Engine::launch_walk(WalkArgs &a, uint64_t walkers, hipStream_t s) {
    // a walk of one source that stays in it reads no table
    a.due.n = 0;
    if (a.span_resident || a.nsrc) {
        if (table_due.n > kTableFew || table_told.n) {
            LT_TRY(flush_tables());
        } else {  // the fix-up behind this walk sets them
            a.due.n = table_due.n;
            for (uint32_t k = 0; k < table_due.n; k++) {
                a.due.part[k] = table_due.part[k];
                a.due.rowptr[k] = table_due.rowptr[k];
                a.due.col[k] = table_due.col[k];
                a.due.words[k] = table_due.words[k];
            }
            table_told = a.due;
            table_due.n = 0;
        }
    }
    const uint64_t fill = (uint64_t)num_cu * 4 * 6 * 64;  // threads for ~6 waves per SIMD
    const int wpt = cfg.walkers_per_thread > 0 ? cfg.walkers_per_thread
                    : walkers >= 4 * fill         ? 4
                    : walkers >= 2 * fill         ? 2
                                                  : 1;
    const uint64_t bw = (uint64_t)kBlock * wpt;
    // with loads going on, room for a pull kernel's workgroups beside the walk's
    const uint64_t most = walk_grid[app_kind][wpt] - (nslots < P && walk_grid[app_kind][wpt] > kPullGrid ? kPullGrid : 0);
    // A batch's queues start a pass each.  (Starting a chunk each, with a grid for the
    // sum of walkers, left sixteen short queues to one workgroup, one after
    // another: 300-450 us a launch, two fifths of the s20 ppr job's time.)
    uint64_t passes = (walkers + bw - 1) / bw;
    if (a.nsrc) {
        a.voff[0] = 0;
        for (uint32_t k = 0; k < a.nsrc; k++) a.voff[k + 1] = a.voff[k] + (counts[a.srcs[k]] + bw - 1) / bw * bw;
        passes = a.voff[a.nsrc] / bw;
    }
    const int grid = (int)std::max<uint64_t>(1, std::min<uint64_t>(passes, most));
    walk_fn(app_kind, wpt, append_gen())<<<grid, kBlock, lds_bytes(wpt), s>>>(a);
    LT_HIP(hipGetLastError());
    meta_dirty = true;
    return LT_OK;
}

// Consume the whole queue of partition p in slices of kSliceChunks chunks:
// walk kernel, then fix-up kernel per slice (processInMemory with all
// batches, src/WalkManager.h:375-388).
lt_status Engine::process(uint32_t p, bool zerocopy, uint64_t walkers) {
    if (spill_on) walkers = dcounts[p];  // counts[p] also holds the walkers spilled to host
    const uint64_t host = spill_on ? hcount[p] : 0;
    if (walkers == 0 && host == 0) return LT_OK;
    WalkArgs a{};
    a.append_mode = cfg.append_mode;
    a.app = app;
    a.q = q;
    a.pt.node_off = d_node_off;
    a.pt.edge_off = d_edge_off;
    a.pt.lut = d_lut;
    a.pt.rec = d_rec;
    a.pt.lut_shift = lut_shift;
    a.pt.P = P;
    a.src = p;
    a.nb = part.node_off[p];
    a.ne = part.node_off[p + 1];
    a.eb = part.edge_off[p];
    a.n = (uint32_t)walkers;
    a.zerocopy = zerocopy ? 1 : 0;
    a.span_resident = cfg.span == LT_SPAN_RESIDENT ? 1 : 0;
    a.stats = d_stats;
    a.ss = sched_state(false);
    if (zerocopy) {
        a.rowptr = zc_rowptr + part.node_off[p];
        a.col = zc_col + part.edge_off[p];
    } else {
        uint64_t *rp;
        uint32_t *cp;
        slot_ptrs(p, &rp, &cp);
        a.rowptr = rp;
        a.col = cp;
        a.words = slot_words(p, cp);
    }
    EventTimer &phase = zerocopy ? t_zc : t_compute;
    hipEvent_t tp = phase.begin(s_compute);
    const uint64_t nch = (walkers + kChunk - 1) / kChunk;
    for (uint64_t lo = 0; lo < nch; lo += slice) {
        const uint64_t hi = std::min<uint64_t>(nch, lo + slice);
        const bool last = hi == nch;
        a.chunk_lo = (uint32_t)lo;
        a.chunk_hi = last ? 0xFFFFFFFFu : (uint32_t)hi;
        const uint64_t sw = std::min<uint64_t>(walkers, hi * kChunk) - lo * kChunk;
        EventTimer &kt = zerocopy ? t_kzc : t_kernel;
        hipEvent_t tk = kt.begin(s_compute);
        LT_TRY(launch_walk(a, sw, s_compute));
        kt.end(tk, s_compute);
        st.zerocopy_launches += zerocopy ? 1 : 0;
        Consumed d{};
        d.n = 1;
        d.src[0] = p;
        d.chunk_lo = (uint32_t)lo;
        d.chunk_hi = a.chunk_hi;
        d.last = last ? 1 : 0;
        LT_TRY(launch_fixup(d));
        st.kernel_launches++;
    }
    if (host) LT_TRY(process_host(p, a));
    phase.end(tp, s_compute);
    return LT_OK;
}

// ---- host walker spill -------------------------------------------------------
lt_status Engine::host_chunk(uint32_t &id) {
    if (hfree.empty()) {
        Walker *b = nullptr, *bd = nullptr;
        LT_HIP(hipHostMalloc((void **)&b, sizeof(Walker) * kChunk * kHostBlockChunks,
                             hipHostMallocMapped | hipHostMallocCoherent));
        hblocks.push_back(b);
        LT_HIP(hipHostGetDevicePointer((void **)&bd, b, 0));
        hblocks_dev.push_back(bd);
        const uint32_t base = (uint32_t)(hblocks.size() - 1) * kHostBlockChunks;
        for (uint32_t k = kHostBlockChunks; k-- > 0;) hfree.push_back(base + k);
    }
    id = hfree.back();
    hfree.pop_back();
    return LT_OK;
}

void Engine::host_reset() {
    for (uint32_t p = 0; p < P; p++) {
        for (uint32_t c : hq[p]) hfree.push_back(c);
        hq[p].clear();
        hhead[p] = hcount[p] = 0;
    }
}

// getEvictedPartition (src/Scheduler.h:149-166): among the partitions other
// than `except` holding at least one full chunk on the device, the one with the
// fewest walkers in all; else any partition with walkers on the device.
int32_t Engine::spill_victim(uint32_t except) const {
    int32_t full = -1, any = -1;
    for (uint32_t i = 0; i < P; i++) {
        if (i == except || dcounts[i] == 0) continue;
        if (dcounts[i] >= kChunk) {
            if (full < 0 || counts[i] < counts[full]) full = (int32_t)i;
        } else if (any < 0 || counts[i] < counts[any]) {
            any = (int32_t)i;
        }
    }
    return full >= 0 ? full : any;
}

// evictWalker (src/Scheduler.h:53-58) for a set of partitions at once: their
// whole device queues go behind their host queues (one gather launch writing
// to mapped host memory), then their chunks return to the pool.  Called with
// the compute stream idle and dcounts fresh.
lt_status Engine::spill_round(const std::vector<uint32_t> &victims) {
    if (victims.empty()) return LT_OK;
    const uint32_t nv = (uint32_t)victims.size();
    std::vector<uint64_t> prefix(nv + 1, 0);
    std::vector<uint32_t> cprefix(nv + 1, 0), hstart(nv), hbase(nv);
    std::vector<Walker *> hptr;
    for (uint32_t k = 0; k < nv; k++) {
        const uint32_t v = victims[k];
        const uint64_t n = dcounts[v], pos = hhead[v] + hcount[v];
        while (((pos + n - 1) >> kChunkLog2) >= hq[v].size()) {
            uint32_t id;
            LT_TRY(host_chunk(id));
            hq[v].push_back(id);
        }
        hstart[k] = (uint32_t)(pos & (kChunk - 1));
        hbase[k] = (uint32_t)hptr.size();
        for (uint64_t c = pos >> kChunkLog2; c <= (pos + n - 1) >> kChunkLog2; c++)
            hptr.push_back(host_chunk_ptr(hq[v][c], true));
        prefix[k + 1] = prefix[k] + n;
        cprefix[k + 1] = cprefix[k] + (uint32_t)((n + kChunk - 1) / kChunk);
    }
    // plan: part | prefix | cprefix | hstart | hbase | hptr, 8-byte aligned pieces
    const size_t o_part = 0, o_prefix = (4 * (size_t)nv + 7) & ~(size_t)7, o_cprefix = o_prefix + 8 * ((size_t)nv + 1);
    const size_t o_hstart = o_cprefix + 4 * ((size_t)nv + 1), o_hbase = o_hstart + 4 * (size_t)nv;
    const size_t o_hptr = (o_hbase + 4 * (size_t)nv + 7) & ~(size_t)7, bytes = o_hptr + 8 * hptr.size();
    if (plan_cap < bytes) {
        dfree(d_plan);
        if (h_plan) (void)hipHostFree(h_plan);
        h_plan = nullptr;
        plan_cap = 0;
        LT_TRY(dmalloc(&d_plan, bytes));
        LT_HIP(hipHostMalloc((void **)&h_plan, bytes, hipHostMallocDefault));
        plan_cap = bytes;
    }
    memcpy(h_plan + o_part, victims.data(), 4 * (size_t)nv);
    memcpy(h_plan + o_prefix, prefix.data(), 8 * ((size_t)nv + 1));
    memcpy(h_plan + o_cprefix, cprefix.data(), 4 * ((size_t)nv + 1));
    memcpy(h_plan + o_hstart, hstart.data(), 4 * (size_t)nv);
    memcpy(h_plan + o_hbase, hbase.data(), 4 * (size_t)nv);
    memcpy(h_plan + o_hptr, hptr.data(), 8 * hptr.size());
    hipEvent_t te = t_wevict.begin(s_compute);
    LT_HIP(hipMemcpyAsync(d_plan, h_plan, bytes, hipMemcpyHostToDevice, s_compute));
    SpillArgs sa{};
    sa.q = q;
    sa.nv = nv;
    sa.part = (const uint32_t *)(d_plan + o_part);
    sa.prefix = (const uint64_t *)(d_plan + o_prefix);
    sa.cprefix = (const uint32_t *)(d_plan + o_cprefix);
    sa.hstart = (const uint32_t *)(d_plan + o_hstart);
    sa.hbase = (const uint32_t *)(d_plan + o_hbase);
    sa.hptr = (Walker *const *)(d_plan + o_hptr);
    const int grid = (int)std::max<uint64_t>(1, std::min<uint64_t>((prefix[nv] + 255) / 256, (uint64_t)num_cu * 8));
    spill_gather_kernel<<<grid, 256, 0, s_compute>>>(sa);
    LT_HIP(hipGetLastError());
    sa.q.seq = ++meta_seq;
    release_queues_kernel<<<1, kBlock, 0, s_compute>>>(sa);
    LT_HIP(hipGetLastError());
    meta_dirty = false;
    meta_seen = false;
    t_wevict.end(te, s_compute);
    LT_TRY(wait_meta());  // the plan and host chunks are final before they are reused
    for (uint32_t k = 0; k < nv; k++) {
        hcount[victims[k]] += dcounts[victims[k]];
        dcounts[victims[k]] = 0;
    }
    st.walker_evicting_calls += nv;
    return LT_OK;
}

// handleWalkerPoolOverflow (src/Scheduler.h:59-82): make room for `want`
// walkers (at least half the capacity when want is larger) by spilling device
// queues, never `except`'s.  Once spilling is needed it goes down to half the
// capacity in one round, so that the reloads that follow do not spill again
// one queue at a time.
lt_status Engine::ensure_room(uint64_t want, uint32_t except, uint64_t &room) {
    const uint64_t target = std::max<uint64_t>(1, std::min<uint64_t>(want, dev_cap / 2));
    LT_TRY(read_meta());
    uint64_t live = 0;
    for (uint32_t i = 0; i < P; i++) live += dcounts[i];
    if (live + target > dev_cap) {
        const uint64_t goal = std::min<uint64_t>(dev_cap - target, dev_cap / 2);
        std::vector<uint64_t> keep(dcounts);  // spill_victim reads dcounts: mark victims by zeroing
        std::vector<uint32_t> victims;
        while (live > goal) {
            const int32_t v = spill_victim(except);
            if (v < 0) break;
            live -= dcounts[v];
            victims.push_back((uint32_t)v);
            dcounts[v] = 0;
        }
        dcounts = keep;
        LT_TRY(spill_round(victims));
        LT_TRY(read_meta());
        live = 0;
        for (uint32_t i = 0; i < P; i++) live += dcounts[i];
        if (live + target > dev_cap) {
            set_error("no walkers left to spill (%llu on the device, capacity %llu)", (unsigned long long)live,
                      (unsigned long long)dev_cap);
            return LT_E_INTERNAL;
        }
    }
    room = std::min<uint64_t>(want, dev_cap - live);
    return LT_OK;
}

// walkerLoadingPhase + computeOffMemory (src/Scheduler.h:215-233,
// src/WalkManager.h:389-421): walk p's spilled walkers in launches of at most
// kMaxHostPieces pieces, read from host memory by the kernel, after making
// room on the device for the walkers they may append.
lt_status Engine::process_host(uint32_t p, const WalkArgs &a) {
    while (hcount[p] > 0) {
        uint64_t room;
        LT_TRY(ensure_room(std::min<uint64_t>(hcount[p], (uint64_t)kMaxHostPieces * kChunk), p, room));
        WalkArgs b = a;
        b.nhost = 0;
        uint64_t pos = hhead[p], total = 0;
        while (b.nhost < kMaxHostPieces && total < room) {
            const uint64_t off = pos & (kChunk - 1);
            const uint64_t len = std::min<uint64_t>(kChunk - off, room - total);
            b.hptr[b.nhost] = host_chunk_ptr(hq[p][pos >> kChunkLog2], true) + off;
            b.hn[b.nhost] = (uint32_t)len;
            b.nhost++;
            pos += len;
            total += len;
        }
        hipEvent_t tl = t_wload.begin(s_compute);
        hipEvent_t tk = t_kernel.begin(s_compute);
        LT_TRY(launch_walk(b, total, s_compute));
        t_kernel.end(tk, s_compute);
        LT_TRY(launch_fixup(Consumed{}));
        t_wload.end(tl, s_compute);
        LT_TRY(wait_meta());  // the pieces go back to the free list below
        hhead[p] += total;
        hcount[p] -= total;
        while (!hq[p].empty() && (hhead[p] >= kChunk || hcount[p] == 0)) {
            hfree.push_back(hq[p].front());
            hq[p].pop_front();
            hhead[p] = hhead[p] >= kChunk ? hhead[p] - kChunk : 0;
        }
        if (hcount[p] == 0) hhead[p] = 0;
        counts[p] = dcounts[p] + hcount[p];
        spill_h2d_bytes += total * sizeof(Walker);
        st.walker_loading_calls++;
        st.kernel_launches++;
    }
    return LT_OK;
}

// Walk the queue of c over PCIe; with zc_batch > 1 also the next largest
// queues below the threshold (not resident, not being copied), in one launch.
lt_status Engine::process_zc(uint32_t c, const uint8_t *pending) {
    std::vector<uint32_t> batch{c};
    if (zc_batch > 1 && !spill_on) {  // a batch consumes device queues only
        std::vector<uint32_t> cand;
        for (uint32_t i = 0; i < P; i++)
            if (i != c && !resident[i] && !(pending && pending[i]) && counts[i] > 0 && counts[i] < zc_threshold)
                cand.push_back(i);
        const size_t take = std::min<size_t>(cand.size(), zc_batch - 1);
        std::partial_sort(cand.begin(), cand.begin() + take, cand.end(), [&](uint32_t x, uint32_t y) {
            return counts[x] != counts[y] ? counts[x] > counts[y] : x < y;
        });
        uint64_t chunks = (counts[c] + kChunk - 1) / kChunk;
        for (size_t k = 0; k < take; k++) {
            const uint64_t ch = (counts[cand[k]] + kChunk - 1) / kChunk;
            if (chunks + ch > slice) break;  // the pool holds at most `slice` consumed chunks per launch
            chunks += ch;
            batch.push_back(cand[k]);
        }
    }
    for (uint32_t p : batch) record(p, 1, -1, -1);
    st.zerocopy_calls += batch.size();
    if (batch.size() == 1) return process(c, true, counts[c]);
    return walk_batch(batch, true);
}

// Walk the queue of the resident partition c (its decision already
// recorded); with resident_batch > 1 also the largest other resident queues
// of at least one chunk, in one launch, each recorded as a decision of the
// same kind.  Partitions brought in by a prefetch and walked here count as
// prefetch hits.
lt_status Engine::process_resident(uint32_t c, int kind, uint8_t *prefetched) {
    std::vector<uint32_t> batch{c};
    uint64_t chunks = (counts[c] + kChunk - 1) / kChunk;
    if (res_batch > 1 && !spill_on && chunks < slice) {
        std::vector<uint32_t> cand;
        for (uint32_t i = 0; i < P; i++)
            if (i != c && resident[i] && counts[i] >= kChunk) cand.push_back(i);
        const size_t take = std::min<size_t>(cand.size(), res_batch - 1);
        std::partial_sort(cand.begin(), cand.begin() + take, cand.end(), [&](uint32_t x, uint32_t y) {
            return counts[x] != counts[y] ? counts[x] > counts[y] : x < y;
        });
        for (size_t k = 0; k < take; k++) {
            const uint64_t ch = (counts[cand[k]] + kChunk - 1) / kChunk;
            if (chunks + ch > slice) break;  // the pool holds at most `slice` consumed chunks per launch
            chunks += ch;
            batch.push_back(cand[k]);
        }
    }
    if (batch.size() == 1) return process(c, false, counts[c]);
    for (size_t k = 1; k < batch.size(); k++) {
        record(batch[k], kind, -1, -1);
        if (prefetched && prefetched[batch[k]]) {
            st.prefetch_hits++;
            prefetched[batch[k]] = 0;
        }
    }
    st.resident_batched += batch.size() - 1;
    return walk_batch(batch, false);
}

// One launch over the whole queues of `parts` (span resident).  Resident
// partitions are in the partition table; of a zero-copy batch the kernel
// knows the members.  (Entered in the table for the launch as well, they cost a
// launch of their own before it.)  Either way a walker that moves between them
// keeps walking, and no queue being consumed is appended to.
lt_status Engine::walk_batch(const std::vector<uint32_t> &parts, bool zerocopy) {
    WalkArgs a{};
    a.append_mode = cfg.append_mode;
    a.app = app;
    a.q = q;
    a.pt.node_off = d_node_off;
    a.pt.edge_off = d_edge_off;
    a.pt.lut = d_lut;
    a.pt.rec = d_rec;
    a.pt.lut_shift = lut_shift;
    a.pt.P = P;
    a.span_resident = 1;
    a.stats = d_stats;
    a.ss = sched_state(false);
    Consumed d{};
    d.n = a.nsrc = (uint32_t)parts.size();
    d.chunk_hi = 0xFFFFFFFFu;
    d.last = 1;
    a.zerocopy = zerocopy ? 1 : 0;
    std::fill(a.srcs, a.srcs + kMaxZcBatch, kEmpty);
    a.src = parts[0];
    uint64_t total = 0;
    for (uint32_t k = 0; k < d.n; k++) {
        const uint32_t p = parts[k];
        d.src[k] = a.srcs[k] = p;
        total += counts[p];
    }
    EventTimer &phase = zerocopy ? t_zc : t_compute;
    EventTimer &kt = zerocopy ? t_kzc : t_kernel;
    hipEvent_t tp = phase.begin(s_compute);
    hipEvent_t tk = kt.begin(s_compute);
    LT_TRY(launch_walk(a, total, s_compute));
    kt.end(tk, s_compute);
    st.zerocopy_launches += zerocopy ? 1 : 0;
    LT_TRY(launch_fixup(d));
    st.kernel_launches++;
    phase.end(tp, s_compute);
    return LT_OK;
}

// One decision: with tracing, the choice and the state it was taken on; then
// a walk from HBM (every kind but 1, zero-copy) advances p's recency.
void Engine::record(uint32_t p, int kind, int32_t loaded, int32_t evicted) {
    if (cfg.record_trace) {
        trace.push_back(lt_trace_rec{(int32_t)p, kind, loaded, evicted, counts[p]});
        for (uint32_t i = 0; i < P; i++) trace_counts.push_back((uint32_t)counts[i]);
        trace_resident.insert(trace_resident.end(), resident.begin(), resident.end());
        for (uint32_t i = 0; i < P; i++) trace_age.push_back(age_of(i));
        int32_t rec[kRecent];
        recent_loads(rec);
        trace_recent.insert(trace_recent.end(), rec, rec + kRecent);
    }
    if (kind != 1) last_use[p] = ++use_clock;
}

uint32_t Engine::age_of(uint32_t p) const {
    return (uint32_t)std::min<uint64_t>(use_clock - last_use[p], 0xFFFFFFFFu);
}

void Engine::recent_loads(int32_t *out) const {
    const auto &h = sched.history;
    for (int k = 0; k < kRecent; k++) out[k] = k < (int)h.size() ? h[h.size() - 1 - k] : -1;
}

// Scores of every partition for the decision that chose `cur`.
lt_status Engine::infer_scores(int32_t cur) {
    scores_valid = false;
    if (!scorer || !scorer_trained(scorer)) return LT_OK;
    LT_TRY(infer_launch(cur));
    return infer_collect();
}

// Launch the inference of the decision that chose `cur` without waiting for
// it (the state is copied at once); infer_collect makes its scores current.
lt_status Engine::infer_launch(int32_t cur) {
    LT_TRY(infer_collect());  // one inference in flight
    if (!scorer || !scorer_trained(scorer)) return LT_OK;
    std::vector<uint32_t> c32(P), a32(P);
    for (uint32_t i = 0; i < P; i++) {
        c32[i] = (uint32_t)std::min<uint64_t>(counts[i], 0xFFFFFFFFu);
        a32[i] = age_of(i);
    }
    DecisionState d;
    d.counts = c32.data();
    d.resident = resident.data();
    d.age = a32.data();
    recent_loads(d.recent);
    d.cur = cur;
    d.w_total = (float)w_run;
    LT_TRY(scorer_infer_launch(scorer, d, nullptr));
    infer_pending = true;
    pending_clock = use_clock;
    return LT_OK;
}

lt_status Engine::infer_collect() {
    if (!infer_pending) return LT_OK;
    infer_pending = false;
    scores_valid = false;
    // another caller of the scorer (after a run that ended early) waited for it
    if (!scorer || !scorer_infer_pending(scorer)) return LT_OK;
    scores.resize((size_t)P * kOut);
    LT_TRY(scorer_infer_wait(scorer, scores.data()));
    scores_clock = pending_clock;
    bool ok = true;
    for (float v : scores) ok = ok && std::isfinite(v);
    scores_valid = ok;
    return LT_OK;
}

// Victim among the resident partitions other than a and b: those with the
// fewest queued walkers; of them the evict_shortlist least recently walked
// (all of them with 0, the default); of those the one with the lowest keep
// score (ties: lowest id).  A shortlist bounds the network's mistakes on
// states unlike its training traces (a network trained on Belady's choices
// for the plain scheduler's states can rank a partition walked moments ago
// lowest on the states its own choices lead to).  Without valid scores, the
// plain rule.
int32_t Engine::learned_victim(int32_t a, int32_t b) {
    if (scores_valid) {
        uint64_t fewest = UINT64_MAX;
        for (uint32_t i = 0; i < P; i++)
            if (resident[i] && (int32_t)i != a && (int32_t)i != b) fewest = std::min(fewest, counts[i]);
        if (fewest != UINT64_MAX) {
            std::vector<std::pair<uint32_t, int32_t>> cand;  // (age, id)
            for (uint32_t i = 0; i < P; i++)
                if (resident[i] && (int32_t)i != a && (int32_t)i != b && counts[i] == fewest)
                    cand.push_back({age_of(i), (int32_t)i});
            const size_t k = cfg.evict_shortlist > 0 ? (size_t)cfg.evict_shortlist : cand.size();
            if (k < cand.size()) {  // oldest first, ties by id
                std::partial_sort(cand.begin(), cand.begin() + k, cand.end(),
                                  [](const std::pair<uint32_t, int32_t> &x, const std::pair<uint32_t, int32_t> &y) {
                                      return x.first > y.first || (x.first == y.first && x.second < y.second);
                                  });
                cand.resize(k);
            }
            int32_t v = -1;
            float keep = 0.f;
            for (const auto &e : cand) {
                const float kv = scores[(size_t)e.second * kOut + 1];
                if (v < 0 || kv < keep || (kv == keep && e.second < v)) {
                    keep = kv;
                    v = e.second;
                }
            }
            sched.learned_decisions++;
            return v;
        }
    }
    sched.fallback_decisions++;
    return lt_sched_evict_min(P, counts.data(), resident.data(), a);
}

// GPUScheduler::run (src/Scheduler.h:311-330) without host walker spill.
lt_status Engine::run_partition(uint32_t p, int32_t &prev_loaded) {
    st.iterations++;
    const uint64_t n = counts[p];
    // shouldZerocopy (src/Scheduler.h:243-252): counts were read this iteration.
    if (!resident[p] && n < zc_threshold) return process_zc(p, nullptr);
    st.explicit_iterations++;
    // graphLoadingPhase (src/Scheduler.h:173-213)
    if (!resident[p]) {
        int32_t evicted = -1;
        if (free_slots.empty()) {
            const int32_t victim = sched.evict_choice(counts.data(), resident.data(), prev_loaded);
            if (victim < 0) {
                set_error("no partition to evict");
                return LT_E_INTERNAL;
            }
            LT_TRY(evict((uint32_t)victim));
            evicted = victim;
        }
        record(p, 3, (int32_t)p, evicted);
        Load load;
        LT_TRY(load_async(p, false, load));
        st.graph_loading_calls++;
        sched.on_load(p);
        if (cfg.pipeline) {
            // compute resident partitions while the copy is in flight
            while (!loaded(load)) {
                LT_TRY(read_meta());
                const int32_t c = sched.computed_choice(counts.data(), resident.data(), (int32_t)p, kRefPage);
                if (c < 0) break;
                st.computing_calls++;
                record((uint32_t)c, 2, -1, -1);
                LT_TRY(process_resident((uint32_t)c, 2, nullptr));
                LT_TRY(wait_meta());
            }
            // the pipelined work changed the queues; p's count is re-read below
            LT_TRY(read_meta());
        }
        LT_TRY(wait_loaded(load));
        LT_TRY(arrived(p));
    } else {
        record(p, 0, -1, -1);
    }
    prev_loaded = (int32_t)p;
    st.computing_calls++;
    return process_resident(p, 0, nullptr);
}

// Scheduler::start (src/Scheduler.h:425-438).
lt_status Engine::scheduler_loop() {
    int32_t prev = -1, prev_loaded = -1;
    bool sync = false;
    sched.begin_run();
    while (true) {
        LT_TRY(read_meta());
        const int32_t c = sched.next(counts.data(), prev, sync);
        if (c == -2) return LT_E_INTERNAL;
        if (c < 0) {
            if (sync) break;
            sync = true;
            continue;
        }
        sync = false;
        prev = c;
        LT_TRY(run_partition((uint32_t)c, prev_loaded));
    }
    return LT_OK;
}

// Learned scheduling.  Decisions follow the plain scheduler (choice, zero-copy
// rule, pipelined compute during a load), with two changes: while the chosen
// partition is walked, the partitions that will need host data next (the
// scorer's best guesses, or with prefetch_plain the largest such queues) are
// copied into slots ahead of time (prefetch), and a victim is the resident
// partition with the fewest queued walkers, ties broken by the lowest keep
// score: trained on Belady's next-use labels, it names the partition needed
// farthest ahead (the plain rule breaks ties by partition id).  Evictions happen only while the compute stream is idle, and
// a prefetched slot joins the resident table only after its copy completed.
lt_status Engine::scheduler_loop_learned() {
    int32_t prev = -1, prev_loaded = -1;
    bool sync = false;
    struct Inflight {
        int32_t part;
        Load load;
    };
    std::vector<Inflight> inflight;         // prefetch copies in copy-stream order
    std::vector<uint8_t> prefetched(P, 0);  // resident because of a prefetch, not yet picked
    std::vector<uint8_t> pending(P, 0);     // being copied by a prefetch
    const uint32_t depth = (uint32_t)std::max(0, cfg.prefetch_depth);
    // Prefetch targets by the plain rule (prefetch_plain 1 and 2): the
    // largest non-resident queues.  With prefetch_plain 1 the victims follow
    // the plain rule too and the scorer is not used (an ablation that
    // isolates what the network adds); with 2 the scorer picks the victims.
    const bool plain_victims = cfg.prefetch_plain == 1;
    const bool plain_targets = cfg.prefetch_plain != 0;
    LT_TRY(infer_collect());
    scores_valid = false;
    sched.begin_run();
    // make completed prefetches resident, in order; with `upto`, wait for it
    auto retire = [&](int32_t upto) -> lt_status {
        while (!inflight.empty()) {
            Inflight f = inflight.front();
            if (upto < 0 && !loaded(f.load)) break;
            LT_TRY(wait_loaded(f.load));
            inflight.erase(inflight.begin());
            pending[f.part] = 0;
            LT_TRY(arrived((uint32_t)f.part));
            if (f.part == upto) break;
        }
        return LT_OK;
    };
    // reference pipelining: walk resident partitions while the copy engine works
    auto pipeline_while_copying = [&](int32_t except, const Load &load) -> lt_status {
        if (!cfg.pipeline) return LT_OK;
        while (!loaded(load)) {
            LT_TRY(read_meta());
            const int32_t p2 = sched.computed_choice(counts.data(), resident.data(), except, kRefPage);
            if (p2 < 0) break;
            st.computing_calls++;
            record((uint32_t)p2, 2, -1, -1);
            LT_TRY(process_resident((uint32_t)p2, 2, prefetched.data()));
            LT_TRY(wait_meta());
        }
        return read_meta();
    };
    while (true) {
        LT_TRY(read_meta());
        LT_TRY(retire(-1));
        LT_TRY(infer_collect());  // the previous decision's scores, computed while its walk ran
        int32_t c = sched.next(counts.data(), prev, sync);
        if (c < 0) {
            if (sync) break;
            sync = true;
            continue;
        }
        // Stick to a prefetched partition (copied or in flight) whose queue is
        // close to the largest: its data is already on the way.
        if (cfg.prefetch_stick_pct > 0 && !resident[c] && !pending[c]) {
            int32_t s2 = -1;
            for (uint32_t i = 0; i < P; i++)
                if ((pending[i] || prefetched[i]) && counts[i] >= zc_threshold && (s2 < 0 || counts[i] > counts[s2]))
                    s2 = (int32_t)i;
            if (s2 >= 0 && counts[s2] * 100 >= counts[c] * (uint64_t)cfg.prefetch_stick_pct) c = s2;
        }
        // The scorer's next partition (learned_next): when c still needs host
        // data, walk instead the highest "next" score among the partitions
        // whose queue is within learned_next % of c's (the greedy rule's
        // exclusion of the previous partition kept).  Scores are the last
        // inference's, normally the previous decision's.
        if (cfg.learned_next > 0 && !plain_victims && !resident[c] && !pending[c] && scorer &&
            scorer_trained(scorer)) {
            if (!scores_recent()) LT_TRY(infer_scores(prev));
            if (scores_valid) {
                int32_t s2 = -1;
                float best = 0.f;
                for (uint32_t i = 0; i < P; i++) {
                    if (counts[i] == 0 || counts[i] * 100 < counts[c] * (uint64_t)cfg.learned_next) continue;
                    if ((int32_t)i == prev && !sync) continue;
                    const float v = scores[(size_t)i * kOut];
                    if (s2 < 0 || v > best) {
                        best = v;
                        s2 = (int32_t)i;
                    }
                }
                if (s2 >= 0 && s2 != c) {
                    st.next_overrides++;
                    c = s2;
                }
            }
        }
        sync = false;
        prev = c;
        st.iterations++;
        bool zc = false;
        if (!resident[c] && !pending[c] && counts[c] < zc_threshold) {
            zc = true;
        } else {
            st.explicit_iterations++;
            if (pending[c]) {
                if (!loaded(inflight.front().load) && inflight.front().part == c)
                    LT_TRY(pipeline_while_copying(c, inflight.front().load));
                LT_TRY(retire(c));
            }
            if (resident[c]) {
                if (prefetched[c]) st.prefetch_hits++;
                prefetched[c] = 0;
                record((uint32_t)c, 0, -1, -1);
            } else {
                LT_TRY(retire(inflight.empty() ? -1 : inflight.back().part));  // the copy engine is in-order
                int32_t evicted = -1;
                if (free_slots.empty()) {
                    if (!scores_recent()) LT_TRY(infer_scores(c));
                    evicted = learned_victim(c, prev_loaded);
                    if (evicted < 0) {
                        set_error("no partition to evict");
                        return LT_E_INTERNAL;
                    }
                    LT_TRY(evict((uint32_t)evicted));
                    prefetched[evicted] = 0;
                }
                record((uint32_t)c, 3, c, evicted);
                Load load;
                LT_TRY(load_async((uint32_t)c, false, load));
                st.graph_loading_calls++;
                sched.on_load((uint32_t)c);
                LT_TRY(pipeline_while_copying(c, load));
                LT_TRY(wait_loaded(load));
                LT_TRY(arrived((uint32_t)c));
            }
            prev_loaded = c;
        }
        // Prefetch the predicted next loads while c is walked.  Slots are
        // freed before the walk is launched (the walk then never reads them),
        // with the scores of the previous decision; the targets are chosen
        // with the scores of this decision, computed while the walk runs.
        size_t want = (plain_victims || (scorer && scorer_trained(scorer))) && inflight.size() < depth
                          ? depth - inflight.size()
                          : 0;
        if (want) {  // no more slots than there are partitions a prefetch may take
            size_t cand = 0;
            for (uint32_t i = 0; i < P && cand < want; i++)
                cand += !resident[i] && !pending[i] && (int32_t)i != c && counts[i] >= zc_threshold;
            want = cand;
        }
        if (want) {
            // the scores of the last inference (normally the previous
            // decision's, computed while its walk ran): no inference here on
            // the critical path unless they are far out of date
            if (!scores_recent() && !plain_victims) LT_TRY(infer_scores(c));
            // copies into the freed slots may start at once: no walk is running, and
            // the next one is launched behind the table updates
            while ((scores_valid || plain_victims) && free_slots.size() < want) {
                const int32_t v = learned_victim(c, -1);
                if (v < 0) break;
                LT_TRY(evict((uint32_t)v));
                prefetched[v] = 0;
            }
        }
        st.computing_calls++;
        LT_TRY(zc ? process_zc((uint32_t)c, pending.data()) : process_resident((uint32_t)c, 0, prefetched.data()));
        // this decision's scores, computed while c is walked: the next
        // decision's victims, and (prefetch_plain 0) this decision's targets
        if (!plain_victims) LT_TRY(infer_launch(c));
        if (want && !free_slots.empty()) {
            if (!plain_targets) LT_TRY(infer_collect());
            while ((scores_valid || plain_targets) && inflight.size() < depth && !free_slots.empty()) {
                int32_t q = -1;
                float best = 0.f;
                for (uint32_t i = 0; i < P; i++) {
                    if (resident[i] || pending[i] || (int32_t)i == c || counts[i] < zc_threshold) continue;
                    // the scorer's guess of the next partition needing host data, or
                    // (plain rule) the largest queue among those partitions
                    const float v = plain_targets ? (float)counts[i] : scores[(size_t)i * kOut];
                    if (q < 0 || v > best) {
                        best = v;
                        q = (int32_t)i;
                    }
                }
                if (q < 0) break;
                Load load;
                LT_TRY(load_async((uint32_t)q, true, load));
                inflight.push_back({q, load});
                pending[q] = 1;
                st.graph_loading_calls++;
                sched.on_load((uint32_t)q);
                st.prefetch_issued++;
                prefetched[q] = 1;
            }
        }
    }
    LT_TRY(retire(inflight.empty() ? -1 : inflight.back().part));
    return infer_collect();
}

SchedState Engine::sched_state(bool device) const {
    SchedState ss{};
    ss.ds = device ? d_ds : nullptr;
    ss.slot_of = d_slot_of;
    ss.part_in_slot = d_part_in_slot;
    ss.resident = d_resident;
    ss.rec = d_rec;
    ss.slots = d_slots;
    ss.slot_bytes = slot_sz;
    ss.nslots = nslots;
    ss.zc_rowptr = zc_rowptr;
    ss.rp_host = rp_resident ? 0 : 1;
    ss.zc_col = zc_col;
    ss.zc_threshold = zc_threshold;
    return ss;
}

// Device-scheduled loop: per iteration decide_kernel (the end of the iteration
// before and the plain greedy rules, in one workgroup), load_kernel (partition copy
// over PCIe by the GPU itself) and walk_kernel, both reading the decision from
// device memory.  kGraphIters iterations are captured once into a hipGraph and the graph is
// relaunched until an iteration finds every queue empty; the host reads one
// record per launch instead of syncing on every decision.
constexpr int kGraphIters = 32;

lt_status Engine::scheduler_loop_device() {
    // host residency -> device mirrors
    std::vector<int32_t> hs(P), hp(nslots);
    for (uint32_t i = 0; i < P; i++) hs[i] = resident[i] ? slot_of[i] : -1;
    for (uint32_t s2 = 0; s2 < nslots; s2++) hp[s2] = part_in_slot[s2];
    LT_HIP(hipMemcpyAsync(d_slot_of, hs.data(), 4 * P, hipMemcpyHostToDevice, s_compute));
    LT_HIP(hipMemcpyAsync(d_part_in_slot, hp.data(), 4 * nslots, hipMemcpyHostToDevice, s_compute));
    LT_HIP(hipMemcpyAsync(d_resident, resident.data(), P, hipMemcpyHostToDevice, s_compute));
    DevSched zero{};
    zero.choice = -1;
    LT_HIP(hipMemcpyAsync(d_ds, &zero, sizeof(zero), hipMemcpyHostToDevice, s_compute));
    LT_HIP(hipStreamSynchronize(s_compute));

    WalkArgs a{};
    a.append_mode = cfg.append_mode;
    a.app = app;
    a.q = q;
    a.pt.node_off = d_node_off;
    a.pt.edge_off = d_edge_off;
    a.pt.lut = d_lut;
    a.pt.rec = d_rec;
    a.pt.lut_shift = lut_shift;
    a.pt.P = P;
    a.span_resident = cfg.span == LT_SPAN_RESIDENT ? 1 : 0;
    a.stats = d_stats;
    a.ss = sched_state(true);
    // walkers per lane of the captured walk launches: the queue sizes are only
    // known on the device, so the grid is the full occupancy grid of that WPT
    const int dwpt = cfg.walkers_per_thread > 0 ? cfg.walkers_per_thread : 1;
    BlockImages bi{};
    bi.img = slot_packed ? d_pk_img : nullptr;
    bi.off = d_pk_off;
    bi.size = d_pk_size;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    LT_HIP(hipStreamBeginCapture(s_compute, hipStreamCaptureModeThreadLocal));
    for (int it = 0; it < kGraphIters; it++) {
        decide_kernel<<<1, kBlock, 0, s_compute>>>(q, a.ss, a.pt, bi);
        load_kernel<<<num_cu, 256, 0, s_compute>>>(d_ds);
        walk_fn(app_kind, dwpt, append_gen())<<<walk_grid[app_kind][dwpt], kBlock, lds_bytes(dwpt), s_compute>>>(a);
    }
    hipError_t ce = hipStreamEndCapture(s_compute, &graph);
    if (ce != hipSuccess) {
        set_error("graph capture failed: %s", hipGetErrorString(ce));
        return LT_E_HIP;
    }
    std::unique_ptr<hipGraph_t, void (*)(hipGraph_t *)> gg(&graph, [](hipGraph_t *x) { (void)hipGraphDestroy(*x); });
    LT_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    std::unique_ptr<hipGraphExec_t, void (*)(hipGraphExec_t *)> ge(&exec,
                                                                    [](hipGraphExec_t *x) { (void)hipGraphExecDestroy(*x); });
    DevSched h{};
    uint64_t launches = 0;
    while (true) {
        LT_HIP(hipGraphLaunch(exec, s_compute));
        launches++;
        LT_HIP(hipMemcpyAsync(&h, d_ds, sizeof(h), hipMemcpyDeviceToHost, s_compute));
        LT_HIP(hipStreamSynchronize(s_compute));
        meta_dirty = true;
        if (h.choice < 0) break;
        if (vregion) LT_TRY(read_meta());  // counts the visit log if it fills up
        if (launches > (1ull << 24)) {
            set_error("device schedule did not drain the queues");
            return LT_E_INTERNAL;
        }
    }
    LT_TRY(read_meta());
    // device residency -> host mirrors
    LT_HIP(hipMemcpy(hs.data(), d_slot_of, 4 * P, hipMemcpyDeviceToHost));
    LT_HIP(hipMemcpy(hp.data(), d_part_in_slot, 4 * nslots, hipMemcpyDeviceToHost));
    LT_HIP(hipMemcpy(resident.data(), d_resident, P, hipMemcpyDeviceToHost));
    free_slots.clear();
    for (uint32_t i = 0; i < P; i++) slot_of[i] = resident[i] ? hs[i] : -1;
    for (int32_t s2 = (int32_t)nslots - 1; s2 >= 0; s2--) {
        part_in_slot[s2] = hp[s2];
        if (hp[s2] < 0) free_slots.push_back((uint32_t)s2);
    }
    st.iterations += h.iterations;
    st.explicit_iterations += h.iterations - h.zc_calls;
    st.graph_loading_calls += h.loads;
    st.zerocopy_calls += h.zc_calls;
    st.computing_calls += h.iterations;
    st.h2d_bytes_explicit += h.h2d_bytes;
    st.h2d_bytes_unpacked += h.h2d_bytes;
    st.kernel_launches += (uint64_t)launches * kGraphIters;
    return LT_OK;
}

// Whether the job can walk the flat arrays: every partition cached, walkers
// allowed to walk through all of them in one launch (span resident with
// batches, or a single partition), all of them on the device at once, and no
// decision trace or append ablation asked for.  Edge numbers have to fit 32 bits.
// Partitions not cached yet are loaded first where the queues would load them
// as well: a job of one partition that is not read in place, or one whose
// walkers start all over the graph, enough for each missing partition to be worth
// a chunk of them and not to be read in place.  Walkers of ppr start at their
// sources and may never see a partition: their jobs load as many as they have
// sources, or the last eighth, which the queues would read in place in every job
// (s20 batched ppr: 3.5 ms a job by queues, 1.65 flat).  By queues, a new engine's first job
// took 0.83 ms on s16 (0.50 so, with no pool of queues to allocate) and 14.4 ms
// on s22 (12.4).
bool Engine::can_run_flat(const RunSpec &rs, uint32_t &missing) const {
    missing = 0;
    if (!flat || g->E > 0xFFFFFFFFull || cfg.record_trace || cfg.append_mode != 0 || spill_on) return false;
    if (P > 1 && (cfg.span != LT_SPAN_RESIDENT || res_batch <= 1)) return false;
    for (uint32_t p = 0; p < P; p++) missing += resident[p] ? 0 : 1;
    if (missing == 0) return true;
    if (P == 1) return rs.total >= zc_threshold;
    if (rs.app == APP_PPR && missing > std::max(P / 8, rs.nq)) return false;
    return rs.total / missing >= std::max<uint64_t>(zc_threshold, kChunk);
}

lt_status Engine::load_missing(ResultHelpers &help) {
    if (pk) {
        Load l;
        for (uint32_t p = 0; p < P; p++)
            if (!resident[p]) LT_TRY(load_async(p, false, l));
    } else {  // a flat cache is laid out as the graph: neighbours in one copy
        hipEvent_t t = t_load.begin(s_copy);
        for (uint32_t p = 0, end; p < P; p = end) {
            end = p + 1;
            if (resident[p]) continue;
            while (end < P && !resident[end]) end++;
            const uint32_t nb = part.node_off[p];
            const uint64_t eb = part.edge_off[p];
            const size_t rbytes = ((size_t)part.node_off[end] - nb + 1) * 8, cbytes = (part.edge_off[end] - eb) * 4;
            LT_HIP(hipMemcpyAsync(flat_rowptr + nb, g->rowptr + nb, rbytes, hipMemcpyHostToDevice, s_copy));
            LT_HIP(hipMemcpyAsync(flat_col + eb, g->col + eb, cbytes, hipMemcpyHostToDevice, s_copy));
            st.h2d_bytes_explicit += rbytes + cbytes;
            st.h2d_bytes_unpacked += rbytes + cbytes;
            for (uint32_t i = p; i < end; i++) {
                slot_of[i] = (int32_t)free_slots.back();
                part_in_slot[free_slots.back()] = (int32_t)i;
                free_slots.pop_back();
                loading++;
            }
        }
        t_load.end(t, s_copy);
    }
    start_results(help, true);
    LT_HIP(hipStreamSynchronize(s_copy));
    for (uint32_t p = 0; p < P; p++) {
        if (resident[p]) continue;
        st.graph_loading_calls++;
        sched.on_load(p);
        LT_TRY(arrived(p));
    }
    return LT_OK;
}

// Eight workgroups per CU: the kernels hold few registers, and the lanes of a
// small job should all have one walker before any has two.
static void launch_flat(const FlatArgs &a, int app, int num_cu, hipStream_t s) {
    const uint64_t n = a.id_hi - a.id_lo;
    const int grid = (int)std::min<uint64_t>((n + kBlock - 1) / kBlock, (uint64_t)8 * num_cu);
    if (app == APP_PAGERANK) flat_walk_kernel<APP_PAGERANK><<<grid, kBlock, 0, s>>>(a);
    else if (app == APP_PPR) flat_ppr_kernel<<<grid, kBlock, 0, s>>>(a);
    else flat_walk_kernel<APP_GENERIC><<<grid, kBlock, 0, s>>>(a);
}

// Walkers of one launch: as many as a queue slice of the default size holds,
// which keeps the per-lane event counts far below 2^32.
constexpr uint64_t kFlatPiece = (uint64_t)kSliceChunks * kChunk;

// The whole job over the flat arrays: walkers are created, walked and finished
// in registers, so the queues are not touched.  Row offsets are read as 32
// bits, which halves the lines that the hot rows take in L2.
lt_status Engine::run_flat(const RunSpec &rs, ResultHelpers &help) {
    if (!rowptr32_set) {  // kept: slots of a flat cache are never evicted
        narrow_rowptr_kernel<<<std::min<int>(8 * num_cu, (int)(V / 256 + 1)), 256, 0, s_compute>>>(
            flat_rowptr, d_rowptr32, (size_t)V + 1);
        LT_HIP(hipGetLastError());
        rowptr32_set = true;
    }
    FlatArgs a{};
    a.app = app;
    a.rowptr = d_rowptr32;
    a.col = flat_col;
    a.stats = d_stats;
    // a launch's visits have to fit the log; walks too long for that count directly
    uint64_t piece = kFlatPiece;
    const uint64_t each = app_kind == APP_PAGERANK ? rs.length : 1, room = (uint64_t)vregion * kLogRegions;
    if (a.app.vlog && room / each < std::min<uint64_t>(rs.total, 1u << 16)) a.app.vlog = nullptr;
    if (a.app.vlog) piece = std::min(piece, room / each);
    // Endpoints and moves of fixed-length walks are written by whole waves:
    // straight into the ring, a launch per buffer, so that they reach the host while
    // the next walkers walk.  (PPR lanes end one by one, and paths are written
    // a word per row: those results stay on the device until the end.)
    const uint32_t nout = (uint32_t)outs.size();
    const bool ring = app_kind == APP_GENERIC && !a.app.paths && nout * rs.total >= kManyOut && ring_cap == kRingLarge;
    constexpr uint32_t kTwo = kRing / 2;  // a launch takes two buffers: its last walkers leave
                                          // the card half idle for some 10 us
    if (ring) piece = 2 * kRingBytes / 4 / nout;
    const auto drain = [&](uint64_t k) -> lt_status {  // launch k's results to the caller
        LT_TRY(wait_ring(k % kTwo));
        const uint64_t n = std::min<uint64_t>(piece, rs.total - k * piece);
        for (uint32_t o = 0; o < nout; o++)
            help.copiers().copy(outs[o].dst + k * piece, h_ring + k % kTwo * 2 * kRingBytes + 4 * o * piece, 4 * n);
        return LT_OK;
    };
    hipEvent_t tp = t_compute.begin(s_compute);
    uint64_t k = 0, drained = 0;
    for (; k * piece < rs.total; k++) {
        a.id_lo = k * piece;
        a.id_hi = std::min<uint64_t>(rs.total, a.id_lo + piece);
        if (ring) {
            for (; drained + kTwo <= k; drained++) LT_TRY(drain(drained));
            uint32_t *at = (uint32_t *)(d_ring + k % kTwo * 2 * kRingBytes) - a.id_lo;
            if (app.endpoints) a.app.endpoints = at;
            if (app.moves_out) a.app.moves_out = at + (app.endpoints ? piece : 0);
        }
        hipEvent_t tk = t_kernel.begin(s_compute);
        launch_flat(a, app_kind, num_cu, s_compute);
        LT_HIP(hipGetLastError());
        t_kernel.end(tk, s_compute);
        st.kernel_launches++;
        if (ring) LT_TRY(mark_ring(k % kTwo));
        if (a.app.vlog) LT_TRY(count_log((uint32_t)((a.id_hi - a.id_lo) * each), 0));
        start_results(help, false);
    }
    t_compute.end(tp, s_compute);
    w_run = rs.total;
    st.iterations = st.explicit_iterations = st.computing_calls = 1;
    st.resident_batched = P - 1;
    for (uint32_t p = 0; p < P; p++) last_use[p] = ++use_clock;
    job_finished = ring;
    if (ring) {
        LT_TRY(finish_job(false));
        for (; drained < k; drained++) {  // the last buffer's copy is behind the walks
            if (drained + 1 == k) LT_TRY(wait_walks());
            LT_TRY(drain(drained));
            walks_over();
        }
    }
    return LT_OK;
}

// Last kernels of a job: its small results and event counters into pinned
// memory; waits for them, and so for the job's walks (large results:
// copy_results does).
lt_status Engine::finish_job(bool small) {
    if (small && !outs.empty()) {
        SmallOut o{};
        o.n = (uint32_t)outs.size();
        o.dst = d_out + kOutData;
        for (uint32_t k = 0; k < o.n; k++) {
            o.src[k] = outs[k].src;
            o.end[k] = (k ? o.end[k - 1] : 0) + (uint32_t)outs[k].words;
        }
        small_out_kernel<<<(o.end[o.n - 1] + 255) / 256, 256, 0, s_compute>>>(o);
    }
    finish_kernel<<<1, kStatSlots, 0, s_compute>>>(d_stats, d_out, d_out + kOutFlag, ++out_seq);
    LT_HIP(hipGetLastError());
    if (!small) return LT_OK;
    LT_TRY(wait_walks());
    const uint32_t *from = h_out + kOutData;
    for (const OutSeg &o : outs) {
        memcpy(o.dst, from, 4 * o.words);
        from += o.words;
    }
    return LT_OK;
}

// Whether finish_kernel has been seen to be over.  The first time that it is ends
// the job's running time, on the host's clock by whichever route it walked.
bool Engine::walks_over() {
    if (!over && __atomic_load_n(h_out + kOutFlag, __ATOMIC_ACQUIRE) == out_seq) {
        over = true;
        t_over = std::chrono::steady_clock::now();
    }
    return over;
}

lt_status Engine::wait_walks() {
    if (!over) LT_TRY(poll_host(h_out + kOutFlag, out_seq, "results"));
    walks_over();
    return LT_OK;
}

// Pinned, mapped memory for a ring, if it can be had.
static bool pin(size_t bytes, uint8_t **h, uint8_t **d) {
    if (hipHostMalloc((void **)h, bytes, hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess) {
        if (hipHostGetDevicePointer((void **)d, *h, 0) == hipSuccess) return true;
        (void)hipHostFree(*h);
    }
    (void)hipGetLastError();
    *h = nullptr;
    return false;
}

// Gets what the job's larger results will want, once the device has something to do:
// threads, and a ring.  Pinning takes 30 to 350 us (at an engine's creation it would
// take them from every engine), and the CPU's first read of each page 1.4 us (0.36 ms a
// MB, by four threads 0.12), which helpers do while the job walks.
//
// Results of 8 MB go faster through a ring of 8 MB than through 2: 10 to 20 MB in 1.58-2.3
// ms a job and 1.66-2.4 (1.9-2.8 by plain copies); so do endpoints of flat walks from 4 MB
// on, which only the large ring takes from the walk itself (6 MB: 0.38 and 0.48 ms);
// fewer do not (3.4 to 5.3 MB: 242-418 us and 256-445, 340-560 by plain copies).  But
// reading 8 MB takes a millisecond, three times some jobs.  So a job with no ring yet
// gets the large one if its loads or rounds cover that (cover); else it comes once
// as many results went through the small one as lose what pinning costs, and is used
// when helpers have read all of it, behind the walks of as many jobs as that takes.
void Engine::start_results(ResultHelpers &help, bool cover) {
    if (help.started) return;
    uint64_t words = 0;
    for (const OutSeg &o : outs) words += o.words;
    if (words > kSmallOut) {
        const bool large = words >= (app_kind == APP_GENERIC && !app.paths ? kManyOut : 2 * kManyOut);
        constexpr uint64_t kRingPays = 8u << 20;  // words: 32 MB, 10 to 18 us a MB
        if (words >= kManyOut) help.most = help_most(4);
        if (!h_ring) {
            if (large && cover && pin(kRingLarge, &h_ring, &d_ring)) ring_cap = kRingLarge;
            else if (pin(kRing * kRingSmall, &h_ring, &d_ring)) ring_cap = kRing * kRingSmall;
        }
        if (large && ring_cap < kRingLarge) {
            ring_words += words;
            if (!h_next && (cover || ring_words >= kRingPays) && !pin(kRingLarge, &h_next, &d_next)) ring_words = 0;
        }
        const size_t use = std::min<uint64_t>(4 * words, ring_cap);
        if (use > ring_seen) {
            help.fresh = h_ring + ring_seen;
            help.fresh_bytes = use - ring_seen;
            ring_seen = use;
        } else if (large && h_next) {
            help.fresh = h_next + next_seen;
            help.fresh_bytes = kRingLarge - next_seen;
            reading_next = true;
        }
    }
    help.start(outs);
}

// The large ring takes over once all of it has been read.  Before a job.
void Engine::swap_ring() {
    if (!h_next || next_seen < kRingLarge) return;
    if (h_ring) (void)hipHostFree(h_ring);
    h_ring = h_next;
    d_ring = d_next;
    ring_cap = ring_seen = kRingLarge;
    h_next = d_next = nullptr;
    next_seen = 0;
}

// The ring buffer is full once the stream gets here.
lt_status Engine::mark_ring(uint32_t slot) {
    mark_kernel<<<1, 1, 0, s_compute>>>(d_out + kOutRing + slot, ++ring_seq[slot]);
    LT_HIP(hipGetLastError());
    return LT_OK;
}

lt_status Engine::wait_ring(uint32_t slot) { return poll_host(h_out + kOutRing + slot, ring_seq[slot], "results"); }

// The results in pieces of a ring buffer's size: kernels fill the next buffers
// while the team copies the oldest one out.
lt_status Engine::copy_results(ResultHelpers &help) {
    if (!ring_cap) {
        LT_TRY(wait_walks());
        for (const OutSeg &o : outs) LT_HIP(hipMemcpy(o.dst, o.src, 4 * o.words, hipMemcpyDeviceToHost));
        return LT_OK;
    }
    uint64_t words = 0;
    for (const OutSeg &o : outs) words += o.words;
    const size_t buf = ring_cap == kRingLarge && words >= 2 * kManyOut ? kRingBytes : kRingSmall;
    std::vector<OutSeg> pieces;
    std::vector<size_t> at;  // place of each in the ring: one behind the other if all fit
    size_t end = 0;
    for (const OutSeg &o : outs)
        for (uint64_t i = 0; i < o.words; i += buf / 4) {
            pieces.push_back({o.dst + i, o.src + i, std::min<uint64_t>(buf / 4, o.words - i)});
            at.push_back(end);
            end += (4 * pieces.back().words + 4095) & ~(size_t)4095;
        }
    if (pieces.size() > kRing)
        for (size_t i = 0; i < at.size(); i++) at[i] = i % kRing * buf;
    for (size_t issued = 0, out = 0; out < pieces.size(); out++) {
        for (; issued < pieces.size() && issued < out + kRing; issued++) {
            fill_ring_kernel<<<64, 256, 0, s_compute>>>(pieces[issued].src, (uint32_t *)(d_ring + at[issued]),
                                                        pieces[issued].words);
            LT_TRY(mark_ring(issued % kRing));
            walks_over();
        }
        LT_TRY(wait_walks());
        LT_TRY(wait_ring(out % kRing));
        help.copiers().copy(pieces[out].dst, h_ring + at[out], 4 * pieces[out].words);
    }
    return LT_OK;
}

lt_status Engine::run(const RunSpec &rs, uint32_t *counts_out, uint32_t *endpoints_out, uint32_t *moves_out) {
    LT_HIP(hipSetDevice(device));
    LT_TRY(drop_loads());
    swap_ring();
    reading_next = false;
    memset(&st, 0, sizeof(st));
    st.cache_slots = nslots;
    spill_h2d_bytes = 0;
    st.h2d_bytes_explicit = pending_h2d;  // the rowptr upload, once
    st.h2d_bytes_unpacked = pending_h2d;
    pending_h2d = 0;
    trace.clear();
    trace_counts.clear();
    trace_resident.clear();
    trace_recent.clear();
    trace_age.clear();
    t_load.reset();
    t_compute.reset();
    t_zc.reset();
    t_wload.reset();
    t_wevict.reset();
    t_kernel.reset();
    t_kzc.reset();
    const uint64_t cap = cfg.num_device_walkers ? std::min<uint64_t>(cfg.num_device_walkers, rs.total) : rs.total;
    // More walkers than the device holds: spill to host queues (the
    // reference's -b); the device-scheduled loop runs them in waves instead.
    spill_on = cap < rs.total && !cfg.device_schedule;
    dev_cap = cap;
    const uint64_t wave = spill_on ? rs.total : cap;
    const bool counting = rs.app != APP_GENERIC && counts_out;
    uint32_t missing;
    bool walk_flat = can_run_flat(rs, missing);
    LT_TRY(ensure_memory(rs, std::max<uint64_t>(cap, 1), counting, endpoints_out != nullptr, moves_out != nullptr,
                         walk_flat));

    app_kind = rs.app;
    app = AppArgs{};
    app.seed = cfg.seed;
    app.V = V;
    app.length = rs.length;
    app.source = rs.source;
    app.counts = counting ? d_counts : nullptr;
    app.counts_stride = count_copies > 1 ? V : 0;
    app.vlog = vregion ? vl.log : nullptr;
    app.vcur = d_vcur;
    app.vcap = vregion;
    q.vcur = vregion ? d_vcur : nullptr;
    app.endpoints = endpoints_out ? d_endpoints : nullptr;
    app.moves_out = moves_out ? d_moves : nullptr;
    app.paths = rs.paths_out ? d_paths : nullptr;
    app.rp_host = rp_resident ? 0 : 1;
    if (rs.app == APP_PAGERANK) app.thresh = prob_threshold(1.0 - (double)0.85f);
    else if (rs.app == APP_PPR) app.thresh = prob_threshold((double)rs.prob);
    if (rs.app == APP_PPR && app.thresh == 0) {
        set_error("ppr stop probability %g rounds to zero", (double)rs.prob);
        return LT_E_ARG;
    }
    if (rs.nq) {
        const size_t need = 12 * (size_t)rs.nq + 8;
        if (query_cap < need) {
            if (h_query) (void)hipHostFree(h_query);
            h_query = nullptr;
            query_cap = 0;
            if (hipHostMalloc((void **)&h_query, need, hipHostMallocDefault) == hipSuccess) query_cap = need;
            else (void)hipGetLastError();
        }
        std::vector<uint64_t> plain(h_query ? 0 : need / 8 + 1);  // pinned memory is short
        uint64_t *off = h_query ? (uint64_t *)h_query : plain.data();
        off[0] = 0;
        for (uint32_t i = 0; i < rs.nq; i++) off[i + 1] = off[i] + rs.q_cnt[i];
        memcpy(off + rs.nq + 1, rs.q_src, 4 * (size_t)rs.nq);
        LT_HIP(hipMemcpyAsync(d_qoff, off, 8 * ((size_t)rs.nq + 1), hipMemcpyHostToDevice, s_compute));
        LT_HIP(hipMemcpyAsync(d_qsrc, off + rs.nq + 1, 4 * (size_t)rs.nq, hipMemcpyHostToDevice, s_compute));
        if (!h_query) LT_HIP(hipStreamSynchronize(s_compute));
        app.q_off = d_qoff;
        app.q_src = d_qsrc;
        app.nq = rs.nq;
    }
    const uint64_t nclear = counting ? (uint64_t)V * count_copies : 0;
    begin_kernel<<<(int)std::min<uint64_t>(8 * num_cu, nclear / 1024 + 2), 256, 0, s_compute>>>(d_counts, nclear, d_stats,
                                                                                             vregion ? d_vcur : nullptr);
    LT_HIP(hipGetLastError());
    // a flat job writes every word of these
    if (moves_out && !walk_flat) LT_HIP(hipMemsetAsync(d_moves, 0, 4 * rs.total, s_compute));
    if (rs.paths_out && !walk_flat)  // columns after an early stop stay 0xFFFFFFFF
        LT_HIP(hipMemsetAsync(d_paths, 0xFF, 4 * (size_t)rs.total * (rs.length + 1), s_compute));
    outs.clear();
    if (counts_out) outs.push_back({counts_out, d_counts, V});
    if (endpoints_out) outs.push_back({endpoints_out, d_endpoints, rs.total});
    if (moves_out) outs.push_back({moves_out, d_moves, rs.total});
    if (rs.paths_out) outs.push_back({rs.paths_out, d_paths, rs.total * ((uint64_t)rs.length + 1)});
    uint64_t out_words = 0;
    for (const OutSeg &o : outs) out_words += o.words;
    const bool small = out_words <= kSmallOut;
    ResultHelpers help;

    double running_ms = 0;
    auto t_walk = std::chrono::steady_clock::now();
    job_finished = over = false;
    if (walk_flat && missing) LT_TRY(load_missing(help));
    if (walk_flat) LT_TRY(run_flat(rs, help));
    for (uint64_t id0 = walk_flat ? rs.total : 0; id0 < rs.total; id0 += wave) {
        const uint64_t id1 = std::min<uint64_t>(rs.total, id0 + wave);
        // createWalkers: untimed, as in the reference (src/LightTraffic.h:33-44)
        reset_queues_kernel<<<1024, 256, 0, s_compute>>>(q, P);
        LT_HIP(hipGetLastError());
        meta_dirty = true;
        InitArgs ia{};
        ia.app = app;
        ia.q = q;
        ia.pt.node_off = d_node_off;
        ia.pt.edge_off = d_edge_off;
        ia.pt.lut = d_lut;
        ia.pt.rec = d_rec;
        ia.pt.lut_shift = lut_shift;
        ia.pt.P = P;
        ia.stats = d_stats;
        host_reset();
        for (uint64_t lo = id0; lo < id1;) {  // with spill, in pieces that fit on the device
            uint64_t n = id1 - lo;
            if (spill_on) LT_TRY(ensure_room(n, kEmpty, n));
            ia.id_lo = lo;
            ia.id_hi = lo + n;
            const int grid = (int)std::min<uint64_t>((n + kBlockWalkers - 1) / kBlockWalkers, (uint64_t)max_grid);
            switch (rs.app) {
                case APP_PAGERANK: init_kernel<APP_PAGERANK><<<grid, kBlock, lds_bytes(), s_compute>>>(ia); break;
                case APP_PPR: init_kernel<APP_PPR><<<grid, kBlock, lds_bytes(), s_compute>>>(ia); break;
                default: init_kernel<APP_GENERIC><<<grid, kBlock, lds_bytes(), s_compute>>>(ia); break;
            }
            LT_HIP(hipGetLastError());
            LT_TRY(launch_fixup(Consumed{}));
            lo += n;
        }
        start_results(help, true);
        LT_TRY(wait_meta());
        const auto t0 = std::chrono::steady_clock::now();
        w_run = id1 - id0;
        if (cfg.device_schedule) LT_TRY(scheduler_loop_device());
        else LT_TRY(cfg.policy == LT_SCHED_LEARNED && (scorer || cfg.prefetch_plain) ? scheduler_loop_learned()
                                                                                   : scheduler_loop());
        const auto t1 = std::chrono::steady_clock::now();
        running_ms += std::chrono::duration<double, std::milli>(t1 - t0).count();
    }
    if (!walk_flat) {
        LT_TRY(read_meta());
        for (uint32_t i = 0; i < P; i++)
            if (counts[i]) {
                set_error("partition %u still holds %llu walkers after the run", i, (unsigned long long)counts[i]);
                return LT_E_INTERNAL;
            }
        t_walk = std::chrono::steady_clock::now();
    }
    // the counts are part of the walk's work, so inside the timed region
    if (vregion && !walk_flat) {
        const uint32_t *cur = &h_meta[P + 4];
        LT_TRY(count_log(0, *std::max_element(cur, cur + kLogRegions)));
    }
    if (count_copies > 1) {
        sum_count_copies_kernel<<<std::max(1, 8 * num_cu), 256, 0, s_compute>>>(d_counts, V);
        LT_HIP(hipGetLastError());
    }
    // reduce (app/pagerank.cu:71-74): results back to the host, untimed but for
    // those that the walks write to the ring
    if (!job_finished) LT_TRY(finish_job(small));
    if (!small && !job_finished) LT_TRY(copy_results(help));
    running_ms += std::chrono::duration<double, std::milli>(t_over - t_walk).count();
    if (reading_next) next_seen += help.mapper.wait();
    outs.clear();
    unsigned long long hs[kNumStats];
    for (int i = 0; i < kNumStats; i++) hs[i] = h_out[2 * i] | (unsigned long long)h_out[2 * i + 1] << 32;
    st.running_ms = running_ms;
    st.moves = hs[ST_MOVES];
    st.teleports = hs[ST_TELEPORTS];
    st.visits = hs[ST_VISITS];
    st.residencies = hs[ST_RESIDENCIES];
    st.zerocopy_moves = hs[ST_ZC_MOVES];
    st.h2d_bytes_zerocopy = hs[ST_ZC_READS] * 64ull + spill_h2d_bytes;
    st.nominal_steps = rs.nominal;
    t_load.collect();
    t_compute.collect();
    t_zc.collect();
    t_kernel.collect();
    t_kzc.collect();
    st.graph_loading_ms = t_load.ms;
    st.computing_ms = t_compute.ms;
    st.zerocopy_ms = t_zc.ms;
    t_wload.collect();
    t_wevict.collect();
    st.walker_loading_ms = t_wload.ms;
    st.walker_evicting_ms = t_wevict.ms;
    st.walk_kernel_ms = t_kernel.ms + t_kzc.ms;
    st.walk_kernel_zc_ms = t_kzc.ms;
    st.learned_decisions = sched.learned_decisions;
    st.fallback_decisions = sched.fallback_decisions;
    return LT_OK;
}

}  // namespace lt

struct lt_engine : lt::Engine {};

using namespace lt;

extern "C" {

lt_status lt_engine_create(const lt_graph *g, const lt_partition *p, const lt_config *cfg, lt_engine **out) {
    if (!g || !p || !out) return LT_E_ARG;
    lt_config c;
    if (cfg) c = *cfg;
    else lt_config_default(&c);
    std::unique_ptr<lt_engine> e(new lt_engine);
    lt_status s = e->init(g, p, &c);
    if (s != LT_OK) return s;
    *out = e.release();
    return LT_OK;
}

void lt_engine_destroy(lt_engine *e) { delete e; }

// Walker ids are 64-bit: w * runs walkers must not wrap.
static bool walkers_fit(uint64_t w, uint32_t runs) {
    if (w > UINT64_MAX / runs) {
        set_error("w * runs = %llu * %u walkers exceed 64-bit walker ids", (unsigned long long)w, runs);
        return false;
    }
    return true;
}

// The termination probability of a PPR walk (app/ppr.cu:22-42), in (0, 1].
static bool prob_ok(float prob) {
    if (!(prob > 0.0f && prob <= 1.0f)) {
        set_error("prob must be in (0, 1] (got %g)", (double)prob);
        return false;
    }
    return true;
}

lt_status lt_run_pagerank(lt_engine *e, uint64_t w, uint32_t l, uint32_t runs, uint32_t *counts_out,
                          uint32_t *endpoints_out) {
    if (!e || w == 0 || runs == 0 || !walkers_fit(w, runs)) return LT_E_ARG;
    RunSpec rs;
    rs.app = APP_PAGERANK;
    rs.total = w * runs;
    rs.length = l;
    rs.nominal = w * (uint64_t)l * runs;
    return e->run(rs, counts_out, endpoints_out, nullptr);
}

lt_status lt_run_ppr(lt_engine *e, uint64_t w, uint32_t source, float prob, uint32_t *counts_out,
                     uint32_t *endpoints_out) {
    if (!e || w == 0 || !prob_ok(prob)) return LT_E_ARG;
    if (source >= e->V) {
        set_error("source %u >= number of vertices %u", source, e->V);
        return LT_E_ARG;
    }
    RunSpec rs;
    rs.app = APP_PPR;
    rs.total = w;
    rs.source = source;
    rs.prob = prob;
    rs.nominal = (uint64_t)((double)w / (double)prob);
    return e->run(rs, counts_out, endpoints_out, nullptr);
}

lt_status lt_run_genericwalk(lt_engine *e, uint64_t w, uint32_t l, uint32_t runs, uint32_t *endpoints_out,
                             uint32_t *moves_out) {
    if (!e || w == 0 || runs == 0 || !walkers_fit(w, runs)) return LT_E_ARG;
    RunSpec rs;
    rs.app = APP_GENERIC;
    rs.total = w * runs;
    rs.length = l;
    rs.nominal = w * (uint64_t)l * runs;
    return e->run(rs, nullptr, endpoints_out, moves_out);
}

lt_status lt_run_genericwalk_paths(lt_engine *e, uint64_t w, uint32_t l, uint32_t runs, uint32_t *paths_out) {
    if (!e || w == 0 || runs == 0 || !paths_out || !walkers_fit(w, runs)) return LT_E_ARG;
    RunSpec rs;
    rs.app = APP_GENERIC;
    rs.total = w * runs;
    rs.length = l;
    rs.nominal = w * (uint64_t)l * runs;
    rs.paths_out = paths_out;
    return e->run(rs, nullptr, nullptr, nullptr);
}

lt_status lt_run_ppr_batch(lt_engine *e, uint32_t nq, const uint32_t *sources, const uint64_t *counts, float prob,
                           uint32_t *endpoints_out) {
    if (!e || nq == 0 || !sources || !counts || !prob_ok(prob)) return LT_E_ARG;
    uint64_t total = 0;
    for (uint32_t i = 0; i < nq; i++) {
        if (sources[i] >= e->V) {
            set_error("query %u source %u >= number of vertices %u", i, sources[i], e->V);
            return LT_E_ARG;
        }
        if (counts[i] > UINT64_MAX - total) {
            set_error("the queries' walk counts exceed 64-bit walker ids");
            return LT_E_ARG;
        }
        total += counts[i];
    }
    if (total == 0) {
        set_error("the queries hold no walks");
        return LT_E_ARG;
    }
    RunSpec rs;
    rs.app = APP_PPR;
    rs.total = total;
    rs.prob = prob;
    rs.q_src = sources;
    rs.q_cnt = counts;
    rs.nq = nq;
    rs.nominal = (uint64_t)((double)total / (double)prob);
    return e->run(rs, nullptr, endpoints_out, nullptr);
}

lt_status lt_device_h2d_bandwidth(uint64_t bytes, uint32_t reps, double *gbps_out) {
    if (bytes == 0 || reps == 0) return LT_E_ARG;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
        (void)hipGetLastError();
        set_error("no HIP device visible");
        return LT_E_NODEVICE;
    }
    uint8_t *h = nullptr, *d = nullptr;
    LT_HIP(hipHostMalloc((void **)&h, bytes, hipHostMallocPortable));
    std::unique_ptr<uint8_t, void (*)(uint8_t *)> gh(h, [](uint8_t *x) { (void)hipHostFree(x); });
    memset(h, 1, bytes);
    LT_TRY(dmalloc(&d, bytes));
    std::unique_ptr<uint8_t, void (*)(uint8_t *)> gd(d, [](uint8_t *x) { (void)hipFree(x); });
    hipStream_t s;
    LT_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    std::unique_ptr<ihipStream_t, void (*)(hipStream_t)> gs(s, [](hipStream_t x) { (void)hipStreamDestroy(x); });
    LT_HIP(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s));  // warm
    LT_HIP(hipStreamSynchronize(s));
    hipEvent_t e0, e1;
    LT_HIP(hipEventCreate(&e0));
    LT_HIP(hipEventCreate(&e1));
    LT_HIP(hipEventRecord(e0, s));
    for (uint32_t r = 0; r < reps; r++) LT_HIP(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s));
    LT_HIP(hipEventRecord(e1, s));
    LT_HIP(hipEventSynchronize(e1));
    float ms = 0;
    LT_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (gbps_out) *gbps_out = (double)bytes * reps / (ms * 1e-3) / 1e9;
    return LT_OK;
}

lt_status lt_device_copy_bandwidth(uint64_t bytes, uint32_t reps, double *gbps_out) {
    if (bytes < 16 || reps == 0) return LT_E_ARG;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
        (void)hipGetLastError();
        set_error("no HIP device visible");
        return LT_E_NODEVICE;
    }
    const uint64_t n16 = bytes / 16;
    uint4 *a = nullptr, *b = nullptr;
    LT_TRY(dmalloc(&a, n16));
    std::unique_ptr<uint4, void (*)(uint4 *)> ga(a, [](uint4 *x) { (void)hipFree(x); });
    LT_TRY(dmalloc(&b, n16));
    std::unique_ptr<uint4, void (*)(uint4 *)> gb(b, [](uint4 *x) { (void)hipFree(x); });
    fill_u32_kernel<<<1024, 256>>>((uint32_t *)a, n16 * 4, 1u);
    copy_probe_kernel<<<4096, 256>>>(a, b, n16);  // warm
    LT_HIP(hipGetLastError());
    LT_HIP(hipDeviceSynchronize());
    hipEvent_t e0, e1;
    LT_HIP(hipEventCreate(&e0));
    LT_HIP(hipEventCreate(&e1));
    LT_HIP(hipEventRecord(e0, nullptr));
    for (uint32_t r = 0; r < reps; r++) copy_probe_kernel<<<4096, 256>>>(a, b, n16);
    LT_HIP(hipEventRecord(e1, nullptr));
    LT_HIP(hipEventSynchronize(e1));
    float ms = 0;
    LT_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (gbps_out) *gbps_out = 2.0 * 16.0 * (double)n16 * reps / (ms * 1e-3) / 1e9;
    return LT_OK;
}

lt_status lt_engine_stats(const lt_engine *e, lt_stats *out) {
    if (!e || !out) return LT_E_ARG;
    *out = e->st;
    return LT_OK;
}

lt_status lt_engine_fetch_partition(lt_engine *e, uint32_t part, uint64_t *rowptr_out, uint32_t *col_out) {
    if (!e || !rowptr_out || !col_out || part >= e->P) {
        lt::set_error("lt_engine_fetch_partition: null argument or partition %u out of range", part);
        return LT_E_ARG;
    }
    return e->fetch_partition(part, rowptr_out, col_out);
}

uint64_t lt_engine_trace_len(const lt_engine *e) { return e ? e->trace.size() : 0; }

lt_status lt_engine_trace_state(const lt_engine *e, uint32_t *counts_out, uint8_t *resident_out, uint32_t *age_out,
                                int32_t *recent_out, uint64_t cap) {
    if (!e) return LT_E_ARG;
    const uint64_t n = std::min<uint64_t>(cap, e->trace.size());
    const size_t P = e->P;
    if (counts_out && n) memcpy(counts_out, e->trace_counts.data(), n * P * sizeof(uint32_t));
    if (resident_out && n) memcpy(resident_out, e->trace_resident.data(), n * P);
    if (age_out && n) memcpy(age_out, e->trace_age.data(), n * P * sizeof(uint32_t));
    if (recent_out && n) memcpy(recent_out, e->trace_recent.data(), n * kRecent * sizeof(int32_t));
    return LT_OK;
}

// Training samples from a traced run.  Decisions are the records of kind 0,
// 1 and 3 (kind 2 = pipelined work inside a load).  Output 0's label is the
// next decision's partition when that decision needed host data (kind 1 or
// 3).  Output 1's label, with use_keep = 1, is each partition's share of the
// walkers processed by all later records, times P; with use_keep = 2 it is
// Belady's quantity, how soon the partition is next needed in HBM: with d
// the number of later records of kind 0, 2 or 3 up to and including its next
// one, 1 - ln(1 + d) / ln(1 + n) (0 when it is never needed again), so that
// evicting the lowest score evicts the partition needed farthest ahead.
lt_status lt_scorer_add_trace(lt_scorer *s_, const lt_engine *e, int32_t use_next, int32_t use_keep,
                              uint64_t *added) {
    if (!s_ || !e) return LT_E_ARG;
    lt::Scorer *s = (lt::Scorer *)s_;
    const uint32_t P = e->P;
    if (scorer_partitions(s) != P) {
        set_error("scorer built for %u partitions, engine has %u", scorer_partitions(s), P);
        return LT_E_ARG;
    }
    const auto &tr = e->trace;
    const size_t n = tr.size();
    if (n == 0) {
        set_error("the engine holds no trace (set record_trace)");
        return LT_E_ARG;
    }
    if (use_keep < 0 || use_keep > 2) {
        set_error("use_keep must be 0, 1 or 2 (got %d)", use_keep);
        return LT_E_ARG;
    }
    // suffix traffic per partition, and the position of each partition's next
    // HBM demand, built from the back
    std::vector<double> future(P, 0.0);
    std::vector<uint64_t> next_demand(P, UINT64_MAX);
    std::vector<std::vector<float>> keep_at(n);
    double total = 0;
    uint64_t demands_after = 0;  // records of kind 0, 2, 3 after position j
    int32_t next_need = -1;
    std::vector<int32_t> next_of(n, -1);
    const double ln_n = log1p((double)n);
    for (size_t j = n; j-- > 0;) {
        const auto &r = tr[j];
        if (r.kind != 2) {
            next_of[j] = next_need;
            keep_at[j].resize(P);
            for (uint32_t q = 0; q < P; q++) {
                if (use_keep == 2) {
                    const double d = next_demand[q] == UINT64_MAX ? -1.0 : (double)(demands_after - next_demand[q] + 1);
                    keep_at[j][q] = d < 0 ? 0.f : (float)(1.0 - log1p(d) / ln_n);
                } else {
                    keep_at[j][q] = total > 0 ? (float)(future[q] / total * P) : 0.f;
                }
            }
            next_need = (r.kind == 1 || r.kind == 3) ? r.partition : -1;
        }
        if (r.kind != 1) {  // needed in HBM at this record; numbered from the back
            demands_after++;
            next_demand[r.partition] = demands_after;
        }
        future[r.partition] += (double)r.walkers;
        total += (double)r.walkers;
    }
    Samples &d = scorer_samples(s);
    uint64_t cnt = 0;
    for (size_t j = 0; j < n; j++) {
        const auto &r = tr[j];
        if (r.kind == 2) continue;
        const bool has_next = use_next && next_of[j] >= 0;
        const bool has_keep = use_keep != 0;
        if (!has_next && !has_keep) continue;
        d.counts.insert(d.counts.end(), e->trace_counts.begin() + j * P, e->trace_counts.begin() + (j + 1) * P);
        d.resident.insert(d.resident.end(), e->trace_resident.begin() + j * P, e->trace_resident.begin() + (j + 1) * P);
        d.age.insert(d.age.end(), e->trace_age.begin() + j * P, e->trace_age.begin() + (j + 1) * P);
        d.recent.insert(d.recent.end(), e->trace_recent.begin() + j * kRecent,
                        e->trace_recent.begin() + (j + 1) * kRecent);
        d.cur.push_back(r.partition);
        d.next.push_back(has_next ? next_of[j] : -1);
        d.w_total.push_back((float)e->w_run);
        d.keep.insert(d.keep.end(), keep_at[j].begin(), keep_at[j].end());
        d.wa.push_back(has_next ? 1.f : 0.f);
        d.wb.push_back(has_keep ? 1.f : 0.f);
        d.n++;
        cnt++;
    }
    if (added) *added = cnt;
    return LT_OK;
}

lt_status lt_engine_set_scorer(lt_engine *e, lt_scorer *s) {
    if (!e) return LT_E_ARG;
    if (s && scorer_partitions((lt::Scorer *)s) != e->P) {  // its state and scores are sized by P
        set_error("scorer built for %u partitions, engine has %u", scorer_partitions((lt::Scorer *)s), e->P);
        return LT_E_ARG;
    }
    LT_TRY(e->infer_collect());  // an inference of the previous scorer still in flight
    e->scores_valid = false;
    e->scorer = (lt::Scorer *)s;
    return LT_OK;
}

lt_status lt_engine_trace(const lt_engine *e, lt_trace_rec *out, uint64_t cap) {
    if (!e || !out) return LT_E_ARG;
    const uint64_t n = std::min<uint64_t>(cap, e->trace.size());
    if (n) memcpy(out, e->trace.data(), n * sizeof(lt_trace_rec));
    return LT_OK;
}

}  // extern "C"
