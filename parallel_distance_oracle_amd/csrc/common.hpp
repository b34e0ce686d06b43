// common.hpp -- shared definitions of the PADO GPU library (gfx950 / MI355X).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "pado_gpu.h"

namespace pado {

constexpr uint32_t kBP = 50;          // BITPARALLEL_SIZE (PARA:45)
constexpr uint32_t kBpdStride = 64;   // bytes per vertex in the bp_dist array (50 distances, kBpNzByte on: below)
// Bytes 51..63 of a vertex's distance line: byte kBpNzByte + l tells which of
// the slots 4l..4l+3 have a nonempty S^-1 (bits 0..3) and S^0 (bits 4..7).
// The queries read the line anyway and skip the sets that it rules out.
constexpr uint32_t kBpNzByte = 51;
constexpr uint32_t kBatch = 1024;     // BATCH_SIZE (PARA:42)
constexpr uint8_t kInf8 = 255;        // SMALLI_MAX (GLB:40)
constexpr uint32_t kHubBits = 24;     // packed label = (hub << 8) | dist
constexpr uint32_t kMaxVertices = 1u << kHubBits;
constexpr uint32_t kEmpty = 0xFFFFFFFFu;
constexpr uint32_t kChunk = 16;       // edges per push work descriptor

// Distance domains of the labeling and query kernels (one templated path):
//  * Hop<false> -- the reference's: u8 hop distances (smalli, GLB:29-40),
//    255 = INF, packed label (hub << 8) | dist, hubs below 2^24, iterations
//    below 255 (the reference's u8 counters wrap there);
//  * Hop<true>  -- wide: 12-bit hop distances in (hub << 12) | dist, 4095 =
//    INF, hubs below 2^20, for graphs whose BFS depth reaches 255 (large
//    grids, road-like graphs).  Bit-parallel distances stay u8 with the BFS
//    stopped at level 254 (farther vertices keep 255: no information in that
//    slot), and the bit-parallel checks skip slots with 255 on either side.
template <bool W>
struct Hop {
    static constexpr uint32_t kBits = W ? 12u : 8u;        // distance bits of a packed label
    static constexpr uint32_t kInf = (1u << kBits) - 1u;   // INF distance; also the iteration limit
    static constexpr uint32_t kMaxN = 1u << (32u - kBits); // vertex ids must stay below this
    using Dist = typename std::conditional<W, uint16_t, uint8_t>::type;  // root-distance table entry
    using Out = typename std::conditional<W, uint16_t, uint8_t>::type;   // query answer
};
constexpr uint32_t kWideMaxVertices = Hop<true>::kMaxN;
// Default grids of the labeling kernels (256-thread blocks): one resident
// round of waves at their occupancy, so a launch with little work ends fast.
constexpr uint32_t kPushGrid = 1024;
constexpr uint32_t kAddGrid = 1024;
// Graphs up to 2^17 vertices rarely have more than a few thousand active
// vertices or candidates per iteration: 256 blocks serve them faster (a 40K
// grid: 0.18 s vs 0.22 s with 1024), and concurrent builds share the chip.
inline uint32_t default_grid(uint32_t n) { return n <= (1u << 17) ? 256u : 1024u; }
// The batch labeling's push and add grids and push descriptor size by
// default, chosen on single batches of an earlier build (R-MAT 20 ef16, median
// of 3: push 768 blocks / add 512 blocks / 8-edge descriptors 0.326 s; 1024 /
// 1024 / 16: 0.356 s; 4-edge descriptors tie with 8).  With batches four at a
// time: 768 / 512 123.1 ms, 512 / 512 130.0, 768 / 256 133.7, 1024 / 512 121.5,
// 768 / 1024 120.3, 1024 / 1024 118.5, 2048 / 2048 121.3; R-MAT 16, 256 / 256:
// 3.50 ms, 768 / 512 3.31.
inline uint32_t default_push_grid(uint32_t n) { return n <= (1u << 17) ? 256u : 768u; }
inline uint32_t default_add_grid(uint32_t n) { return n <= (1u << 17) ? 256u : 512u; }
constexpr uint32_t kPushChunk = 8;

// Thread-local error text behind pado_gpu_last_error().
void set_error(const std::string &msg);
void clear_error();

// Status-returning HIP check for the C ABI implementation.
#define PADO_HIP(call)                                                              \
    do {                                                                            \
        hipError_t e_ = (call);                                                     \
        if (e_ != hipSuccess) {                                                     \
            ::pado::set_error(std::string(#call) + ": " + hipGetErrorString(e_));   \
            return PADO_GPU_ERR_HIP;                                                \
        }                                                                           \
    } while (0)

#define PADO_TRY(call)                                  \
    do {                                                \
        pado_gpu_status s_ = (call);                    \
        if (s_ != PADO_GPU_OK) return s_;               \
    } while (0)

// Serialises device allocation and release with hipGraph capture: builds of a
// many-graph job run on several threads, and a release may synchronise the
// device while another thread's stream is capturing.
inline std::recursive_mutex &capture_mutex()
{
    static std::recursive_mutex m;
    return m;
}

// The query copy's record of a vertex: everything about it that a query reads
// but its sets and labels, in one 128-byte line (a weighted index has the
// last four words only):
//   bytes   0..63   the distance line (distances, nonempty-set bits)
//   bytes  64..113  per slot the eight bytes of S^-1 OR-ed into one: two
//                   vertices' sets can meet only where these bytes do
//   word  29        component: vertices with different values are in different
//                   components; 0 throughout an imported index
//   words 30, 31    first label << 24 | label count
constexpr uint32_t kQRecWords = 32, kQRecFold = 16, kQRecTail = 28;
constexpr uint32_t kWRecWords = 4;
constexpr uint32_t kListAlign = 32;  // label list alignment: one 128-byte line

// Temporary device memory of one context's calls, kept from one call for the
// next: a build of R-MAT 20 spent 15 ms of 152 in hipMalloc and hipFree, and
// memory that goes back to the driver is cleared before it is handed out again
// (a build now and then took 300 ms longer once the card's memory had gone
// round).  Everything that takes blocks from it uses them on the context's
// stream only, so a block given back while that stream still works on it is
// safe with the next taker.  What lies idle in it is bounded: a sixteenth of
// the card while a graph of the context lives (it may be built again), else
// kIdleWork, and a sixteenth of the card for all contexts of a device
// together.  All of it goes back when the context is destroyed, when its user
// asks for it (pado_gpu_ctx_trim) and whenever an allocation fails.  Safe with
// several threads.
class WorkPool {
public:
    WorkPool(int device, size_t card_bytes);
    ~WorkPool();
    // A block of at least `bytes` bytes (its size in *got), or null.
    void *take(size_t bytes, size_t *got);
    void give(void *p, size_t bytes);
    // Page-locked host memory of kPinned bytes, or null.
    void *take_pinned();
    void give_pinned(void *p);
    void hold(int graphs);  // graphs of the context that live, more or fewer
    void collect(size_t keep, std::vector<void *> *out);  // takes out idle blocks, oldest first
    void trim();                                          // gives all idle blocks back
    void close();                                         // the context is gone
    void set_limit(size_t bytes);                         // most bytes in use at once (0: any)
    struct Sizes {
        size_t in_use, peak, idle;  // peak: of in_use, since the last trim
    };
    Sizes sizes();
    static constexpr size_t kPinned = 131072;

private:
    struct Block {
        void *p;
        size_t bytes;
    };
    std::mutex mu_;
    std::vector<Block> idle_;  // in the order they were given back
    std::vector<void *> pinned_;
    size_t idle_bytes_ = 0, in_use_ = 0, peak_ = 0, max_use_ = 0, card_bytes_ = 0;
    int device_ = 0, graphs_ = 0;
    bool closed_ = false;
    size_t shared_limit() const;  // idle bytes of all the device's pools
    size_t limit() const;         // of this one
};

// hipMalloc under capture_mutex; where it fails, what the process's pools hold
// idle goes back and it is tried once more.
hipError_t device_alloc(void **p, size_t bytes);

// Device buffer owned by a handle or, with a pool, by a call.  kBufSlack bytes
// past its end are its own too: a 16-byte read that starts inside it may run
// over the end (query.hip).
constexpr size_t kBufSlack = 16;
template <class T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    pado_gpu_status alloc(size_t count, WorkPool *pool = nullptr)
    {
        release();
        if (count == 0) count = 1;
        const size_t bytes = count * sizeof(T) + kBufSlack;
        if (pool) {
            p = static_cast<T *>(pool->take(bytes, &held_));
            pool_ = p ? pool : nullptr;
        } else if (device_alloc((void **)&p, bytes) != hipSuccess) {
            p = nullptr;
        }
        if (!p) {
            set_error("hipMalloc(" + std::to_string(count * sizeof(T)) + " B): out of memory");
            return PADO_GPU_ERR_NOMEM;
        }
        n = count;
        return PADO_GPU_OK;
    }
    void release()
    {
        if (p && pool_) {
            pool_->give(p, held_);
        } else if (p) {
            std::lock_guard<std::recursive_mutex> g(capture_mutex());
            (void)hipFree(p);
        }
        p = nullptr;
        n = 0;
        pool_ = nullptr;
    }
    void swap(DevBuf &o)
    {
        std::swap(p, o.p);
        std::swap(n, o.n);
        std::swap(pool_, o.pool_);
        std::swap(held_, o.held_);
    }
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }

private:
    WorkPool *pool_ = nullptr;
    size_t held_ = 0;  // the pool block's bytes
};

// A call's page-locked T, written by copies on stream st: they are done before
// it goes back.
template <class T>
struct PinnedBuf {
    static_assert(sizeof(T) <= WorkPool::kPinned);
    T *p = nullptr;
    pado_gpu_status alloc(WorkPool *pool, hipStream_t st)
    {
        p = static_cast<T *>(pool->take_pinned());
        if (!p) {
            set_error("hipHostMalloc failed");
            return PADO_GPU_ERR_NOMEM;
        }
        pool_ = pool;
        st_ = st;
        return PADO_GPU_OK;
    }
    PinnedBuf() = default;
    PinnedBuf(const PinnedBuf &) = delete;
    PinnedBuf &operator=(const PinnedBuf &) = delete;
    ~PinnedBuf()
    {
        if (!p) return;
        (void)hipStreamSynchronize(st_);
        pool_->give_pinned(p);
    }

private:
    WorkPool *pool_ = nullptr;
    hipStream_t st_ = nullptr;
};

// The first active lane's value, in scalar registers: for values that are the
// same in every lane (loaded from one address, or broadcast), so that the
// compiler treats them as wave-uniform.
__device__ inline uint64_t uniform64(uint64_t x)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
}

__device__ inline uint32_t uniform32(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

// Lane `lane`'s 64 bits, in scalar registers.  (The builtin returns an int,
// whose sign must not spread over the upper half.)
__device__ inline unsigned long long readlane64(unsigned long long x, uint32_t lane)
{
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)x, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(x >> 32), lane);
    return ((unsigned long long)hi << 32) | lo;
}

// Orders LDS writes of some lanes of a wave before reads by other lanes of the
// same wave.
__device__ inline void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <int CTRL, int ROWS>
__device__ inline uint32_t dpp0(uint32_t x)  // x moved by DPP, 0 where nothing moves in
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xF, false);
}

// Inclusive prefix sum over the 64 lanes of a wave (all of them active): four
// shifts inside the rows of sixteen lanes, then the row totals passed on.  Six
// dependent adds in registers where shuffles were six LDS round trips.
__device__ inline uint32_t wave_incl_scan(uint32_t x)
{
    x += dpp0<0x111, 0xF>(x);
    x += dpp0<0x112, 0xF>(x);
    x += dpp0<0x114, 0xF>(x);
    x += dpp0<0x118, 0xF>(x);
    x += dpp0<0x142, 0xA>(x);
    x += dpp0<0x143, 0xC>(x);
    return x;
}

__device__ inline uint32_t wave_total(uint32_t x) { return __builtin_amdgcn_readlane(wave_incl_scan(x), 63); }

// The wave's OR of x.
__device__ inline uint32_t wave_or(uint32_t x)
{
    x |= dpp0<0x111, 0xF>(x);
    x |= dpp0<0x112, 0xF>(x);
    x |= dpp0<0x114, 0xF>(x);
    x |= dpp0<0x118, 0xF>(x);
    x |= dpp0<0x142, 0xA>(x);
    x |= dpp0<0x143, 0xC>(x);
    return __builtin_amdgcn_readlane(x, 63);
}

// Adds the wave's sums of the lanes' counts x to entries FIRST .. FIRST + N -
// 1 of the wave's row of statistics: kStatRows rows of one 128-byte line each,
// summed once at the end of a build.  A row has few writers and nobody reads
// it during the build: with all waves adding to one set of totals, the queue
// on their line was 4.7 us of the average batch kernel (R-MAT 20 build: 317
// ms, 292 without the totals).  With the rows, the scans by DPP and the
// working counters on lines of their own: 250 ms; a 161 x 161 wide grid 80 ->
// 64.6 ms.
constexpr uint32_t kStatRows = 1024, kStatCols = 16;
template <int FIRST, int N>
__device__ inline void add_stats(unsigned long long *rows, uint32_t wave, const uint32_t (&x)[N])
{
    static_assert(FIRST + N <= (int)kStatCols, "an entry per count");
    const uint32_t lane = threadIdx.x & 63;
    unsigned long long mine = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        // (each half's total fits 32 bits)
        const unsigned long long s = wave_total(x[i] & 0xFFFFu) + ((unsigned long long)wave_total(x[i] >> 16) << 16);
        if (lane == (uint32_t)i) mine = s;
    }
    if (mine) atomicAdd(&rows[(uint64_t)(wave % kStatRows) * kStatCols + FIRST + lane], mine);
}

// Append one item per lane with `pred` to a list counted by *counter: the
// active lanes of the wave take consecutive slots with a single atomic, so a
// shared counter sees one update per wave instead of one per item.  Returns
// the lane's slot (meaningless where !pred).
__device__ inline uint32_t wave_append(uint32_t *counter, bool pred)
{
    const unsigned long long m = __ballot(pred);
    if (m == 0ull) return 0u;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t leader = (uint32_t)__ffsll(m) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = __shfl(base, leader);
    return base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
}

// wave_append through 64 words of LDS of the wave's own, `held` of them in use
// (0 at first): a list that every wave of a large launch adds to sees one
// update per 64 entries or so.  Updates of one word go one after the other,
// some 10 ns each (builds of R-MAT 20: 131.0 -> 128.7 ms, weighted 496 -> 477).
// list_flush puts the rest on the list at the end.
__device__ inline void list_flush(uint32_t *counter, uint32_t *list, const uint32_t *buf, uint32_t &held)
{
    if (held == 0u) return;
    const uint32_t lane = threadIdx.x & 63;
    wave_lds_sync();
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(counter, held);
    base = uniform32(base);
    if (lane < held) list[base + lane] = buf[lane];
    held = 0;
    __builtin_amdgcn_wave_barrier();  // (the next entries must not overtake these reads)
}

__device__ inline void list_append(uint32_t *counter, uint32_t *list, uint32_t *buf, uint32_t &held, bool pred,
                                   uint32_t item)
{
    const unsigned long long m = __ballot(pred);
    if (m == 0ull) return;
    const uint32_t more = (uint32_t)__popcll(m);
    if (held + more > 64u) list_flush(counter, list, buf, held);
    if (pred) buf[held + (uint32_t)__popcll(m & ((1ull << (threadIdx.x & 63)) - 1ull))] = item;
    held += more;
}

// Device-side counters shared by the labeling kernels (one struct per build,
// the statistics rows of add_stats behind it).  Counters that a kernel's waves update
// lie on lines of their own: updates of one line queue behind each other.
struct BuildCounters {
    // Device-side schedule: the batch step reads its parameters from here, so
    // one launch sequence (or one captured hipGraph) serves every batch.
    uint32_t n_vert;       // vertices of the graph
    uint32_t abits_words;  // 64-bit words of one frontier bitmap slot
    uint32_t pull;         // the frontier's push edges are wanted (n_pedge)
    // Batch gate: a batch enqueued before the host has seen the previous one
    // finish runs as no-ops if the previous batch still has a frontier.
    uint32_t hold;         // set: every batch kernel returns at once
    uint32_t iter_last;    // last iteration k_push ran (not held)
    uint32_t next_batch;          // batch index the next k_batch_begin starts
    uint32_t rs, rsz, gen_batch;  // current batch: roots [rs, rs + rsz)
    uint32_t domain;              // an iteration reached 255 (u8 domain)
    // Live iterations summed over batches of 1,024 roots (a batch of 4,096
    // counts for each quarter that has active vertices), and over batches as
    // they are run.
    unsigned long long iterations, steps;
    unsigned long long pulls;     // iterations run in pull form (statistic)
    // Frontier and candidate counts of batch iteration i live in slot i & 1:
    // each kernel reads its own slot and empties the other one for the next
    // kernel to fill, so no control launch runs between iterations.
    alignas(128) uint32_t n_act[2][4];  // nonzero: the iteration has active vertices (of that quarter)
    alignas(128) uint32_t n_chunk[2];  // push work descriptors of the iteration
    alignas(128) uint32_t n_cand[2];   // candidate vertices of the iteration
    alignas(128) uint32_t n_touched;   // vertices whose indicator row was touched this batch
    alignas(128) unsigned long long pool_top;  // next free label slot in the pool
    uint32_t overflow;     // label pool exhausted
    alignas(128) unsigned long long n_pedge[2];  // push edges of the iteration's frontier (sum of push degrees)
    // Statistics: the sums of the rows' entries (k_fold_stats).
    alignas(128) unsigned long long edges;  // push edges scanned (tails >= roots_start)
    unsigned long long tails;     // distinct tails with a fresh indicator bit, summed over iterations
    unsigned long long pushes;    // (tail, root) pairs offered by push
    unsigned long long ind_pass;  // pairs that set a fresh indicator bit
    unsigned long long bp_pruned; // pairs pruned by the bit-parallel check
    unsigned long long cands;     // (vertex, root) candidates after the BP check
    unsigned long long dq_labels; // labels with dist < iter read by distance queries
    unsigned long long dq_pruned; // candidates pruned by the distance query
    unsigned long long labels;    // labels appended
    unsigned long long dq_rows;   // root-distance rows scanned
    unsigned long long actives;   // active vertices, summed over iterations
};
constexpr uint32_t kStats = 11;  // the last fields, in the order of a row's entries
static_assert(kStatRows * kStatCols * 8 % sizeof(BuildCounters) == 0, "rows are allocated in units of the struct");

// Host-side timing of the labeling kernels (HIP events on the build stream).
struct KernelTimes {
    double ms_push = 0, ms_add = 0, ms_bp = 0;
    uint64_t n_push = 0, n_add = 0, n_bp = 0;
};

}  // namespace pado

// Opaque handle definitions (C ABI types).
struct pado_gpu_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t side = nullptr;       // second stream of chunked host-array queries
    hipEvent_t side_ev = nullptr;     // orders the side stream after work queued before a query
    int num_cu = 0;
    bool concurrent = false;          // one of several contexts whose builds run at once (a many-graph job)
    std::shared_ptr<pado::WorkPool> work;  // temporaries of calls on `stream`
};

struct pado_gpu_graph {
    explicit pado_gpu_graph(pado_gpu_ctx *c) : ctx(c), work(c->work) { work->hold(1); }
    ~pado_gpu_graph() { work->hold(-1); }
    pado_gpu_graph(const pado_gpu_graph &) = delete;
    pado_gpu_graph &operator=(const pado_gpu_graph &) = delete;
    pado_gpu_ctx *ctx = nullptr;
    std::shared_ptr<pado::WorkPool> work;  // (a graph may outlive its context)
    uint32_t n = 0;
    uint64_t m = 0;  // directed edge count (2x undirected)
    pado::DevBuf<uint64_t> off;
    pado::DevBuf<uint32_t> adj;
    pado::DevBuf<uint8_t> w;  // edge weights (weighted graphs), else empty
    bool weighted = false;
    std::vector<uint64_t> h_off;  // host copy: root selection is a serial pass
    std::vector<uint32_t> h_adj;
    std::vector<uint8_t> h_w;
};

struct pado_gpu_index {
    pado_gpu_ctx *ctx = nullptr;
    uint32_t n = 0;
    uint32_t weighted = 0;
    uint32_t wide = 0;  // labels in the wide hop domain (Hop<true>)
    uint32_t bp_pass_through = 0;  // wide build whose bit-parallel BFS was cut at level 254:
                                   // its bit-parallel vertices were labeled as ordinary hubs
    // Weighted build: batches held for the host, label pools grown, most words taken of one.
    uint64_t holds = 0, grows = 0, pool_words = 0;
    // Bit-parallel labels, rank space: bpd[v*64 + i], bps[(v*50 + i)*2 + {0,1}];
    // the rest of a bpd line holds the nonempty-set bits (kBpNzByte).
    pado::DevBuf<uint8_t> bpd;
    pado::DevBuf<uint64_t> bps;
    // Canonical labels, rank space: CSR of packed (hub << 8) | dist, hubs ascending.
    pado::DevBuf<uint64_t> loff;
    pado::DevBuf<uint32_t> lab;
    uint64_t num_labels = 0;
    // Weighted labels (hub u32, dist u32), rank space.
    pado::DevBuf<uint32_t> whub;
    pado::DevBuf<uint32_t> wdist;
    // Query copy in original-id order (order_labels, PARA:2198-2281): records
    // (kQRecWords above), sets, and label lists that start at multiples of
    // kListAlign entries and are padded to them with all-ones.
    int ordered = 0;
    int built = 0;  // labeled by this library (not imported): components are known
    pado::DevBuf<uint32_t> qrec;
    pado::DevBuf<uint64_t> qbps;
    pado::DevBuf<uint32_t> qlab;  // packed labels, or hubs of a weighted index
    pado::DevBuf<uint32_t> qwdist;
    // Staging for host-pointer queries.
    pado::DevBuf<uint32_t> qa, qb;
    pado::DevBuf<uint8_t> qout;
    pado::DevBuf<uint32_t> qout32;
    // One-pair queries: the answer word in mapped host memory, the kernel's
    // result slot (pado_gpu_query_pair); its lock serialises callers.
    uint32_t *pair_out = nullptr;
    uint32_t *pair_out_dev = nullptr;
    std::mutex pair_mu;
    ~pado_gpu_index()
    {
        if (pair_out) {
            std::lock_guard<std::recursive_mutex> g(pado::capture_mutex());
            (void)hipHostFree(pair_out);
        }
    }
    // Build statistics.
    double ms_bp = 0, ms_batch = 0, ms_final = 0;
    uint32_t bp_roots[pado::kBP] = {0};
    uint32_t bp_max_level = 0;
    uint64_t iterations = 0;
    pado::BuildCounters counters{};
    pado::KernelTimes ktimes{};
};
