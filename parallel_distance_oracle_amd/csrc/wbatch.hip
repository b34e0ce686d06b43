// wbatch.hip -- weighted pruned landmark labeling on gfx950.
//
// Reference: WeightedParaVertexCentricPLL<512>, includes/pado_weighted_unv_para.h
// (initialize_tables :305-383, send_messages :435-522, distance_query
// :527-914, filter_out_labels :1100-1228, reset_tables :918-956,
// update_index :961-990, vertex_centric_labeling_in_batches :1231-1566).
//
// The reference's labels are the canonical pruned landmark labels: (r, d) is
// a label of v iff r ranks at or above v, d = d(v, r), and no vertex ranked
// above r lies on a shortest v-r path.  Its schedule (queue orders, first
// witness returned by the distance query, in-place filtering) does not change
// that set, and this build reaches the same set with a schedule-free scheme,
// per batch of roots:
//   1. Bellman-Ford rounds from all batch roots at once.  A root's distance
//      travels only to lower-ranked tails (send_messages, WPARA:457-470); a
//      (tail, root) value that improves is checked against the labels of
//      earlier batches (distance_query's first loop, WPARA:569-580): if a
//      2-hop path through an earlier hub is as short, the pair is marked
//      pruned and does not propagate.  Rounds end when nothing improves.
//   2. Filter (filter_out_labels): a surviving pair (v, r) is dropped if some
//      batch root h < r has surviving pairs (v, h), (r, h) with
//      S(v,h) + S(r,h) <= S(v,r).
// Why this is exact: a canonical pair's shortest paths avoid every vertex
// ranked above r, so the restricted search finds d(v,r) and no earlier hub can
// prune it; a non-canonical pair has some higher vertex on a shortest path,
// and the highest such vertex h* either belongs to an earlier batch (then the
// earlier labels prune the pair at any value >= d) or to this batch (then
// (v,h*) and (r,h*) are canonical, exact, and witness the filter).
//
// Layout per batch (B = 512 roots): T[n][B] u32 tentative distances, P and I
// bitmaps (pruned at the current value / improved this round) [n][B/64] u64,
// the earlier-batch root-distance table (hmin[n], dcw[hub][B] u32), and the
// frontier as (vertex, root bitmap) entries with 16-edge push chunks.  Labels
// are packed u64 (hub << 32 | dist) in per-vertex growable arrays.
#include <cstring>

#include "internal.hpp"

namespace pado {
namespace {

constexpr uint32_t kWB = 512;         // roots per batch (WPARA BATCH_SIZE)
constexpr uint32_t kWW = kWB / 64;    // 64-bit words per root bitmap
constexpr uint32_t kWInf = 0xFFFFFFFFu;
using u64 = unsigned long long;

// Frontier / improved-tail counts of round i live in slot i & 1: each round's
// kernels read their slot and empty the other one for the next kernel.
// Counters that a kernel's waves update lie on lines of their own; add_stats'
// rows follow the struct (with the scans by DPP, weighted R-MAT 20: 719 -> 627
// ms; the filter of a late batch, 2,048 blocks of which most are idle, 11.5 ->
// 6.6 us).
struct WCounters {
    uint32_t n_act[2];              // nonzero: the round has active vertices
    u64 rounds;
    uint32_t hold;                  // a batch is not done: nothing after it runs (k_w_filter)
    alignas(128) uint32_t a_top[2];    // active-list slots handed out (per-wave reservations)
    alignas(128) uint32_t n_chunk[2];
    alignas(128) uint32_t n_imp[2];
    alignas(128) uint32_t n_touched;
    alignas(128) u64 pool_top;
    uint32_t overflow;
    // Pool words the batch's commit can reserve at most: per touched vertex
    // the reservation its list would take if every batch root were kept.
    alignas(128) u64 need_bound;
    alignas(128) u64 need, labels;
    // Statistics: the sums of the rows' entries (k_w_fold_stats).
    alignas(128) u64 relax, improved, pruned, filtered;
};
constexpr uint32_t kWStats = 4;

// What the host learns of a batch (in page-locked memory).
struct WClosed {
    u64 rounds;
    uint32_t held, n_touched;
};
constexpr uint32_t kWRing = 4;
struct WHost {
    WCounters c;
    WClosed ring[kWRing];
};

struct WStore {
    u64 *pool;
    u64 *base;
    uint32_t *len, *cap;
    u64 pool_size;
};

__device__ inline uint32_t lane_id() { return threadIdx.x & 63; }

__device__ inline u64 *stat_rows(WCounters *C) { return reinterpret_cast<u64 *>(C + 1); }

__device__ inline uint32_t wave_max(uint32_t x)
{
    x = max(x, dpp0<0x111, 0xF>(x));
    x = max(x, dpp0<0x112, 0xF>(x));
    x = max(x, dpp0<0x114, 0xF>(x));
    x = max(x, dpp0<0x118, 0xF>(x));
    x = max(x, dpp0<0x142, 0xA>(x));
    x = max(x, dpp0<0x143, 0xC>(x));
    return __builtin_amdgcn_readlane(x, 63);
}

// Tails > lo form a prefix of a descending adjacency list (WPARA:457 breaks
// at the first tail <= roots_start).
__device__ inline uint32_t prefix_above(const uint64_t *off, const uint32_t *adj, uint32_t v, uint32_t lo)
{
    const uint32_t lane = lane_id();
    const uint64_t base = off[v];
    uint32_t a = 0, b = (uint32_t)(off[v + 1] - base);
    while (b - a > 64) {
        uint32_t step = (b - a + 63) / 64;
        uint32_t pos = a + lane * step;
        bool p = pos < b && adj[base + pos] > lo;
        uint32_t c = (uint32_t)__popcll(__ballot(p));
        if (c == 0) {
            b = a;
        } else {
            uint32_t na = a + (c - 1) * step + 1, nb = a + c * step;
            a = na;
            if (nb < b) b = nb;
        }
    }
    uint32_t pos = a + lane;
    bool p = pos < b && adj[base + pos] > lo;
    return a + (uint32_t)__popcll(__ballot(p));
}

// Pool words a commit of up to `add` new labels may reserve for a list of
// length len and capacity cap (lists double).
__device__ inline u64 reserve_words(uint32_t len, uint32_t cap, uint32_t add)
{
    if (len + add <= cap) return 0;
    uint32_t ncap = cap * 2;
    if (ncap < len + add) ncap = len + add;
    if (ncap < 8) ncap = 8;
    return ncap;
}

// The statistics rows' sums into the totals (once, at the end).
__global__ __launch_bounds__(1024) void k_w_fold_stats(WCounters *C)
{
    __shared__ u64 s[kStatCols];
    if (threadIdx.x < kStatCols) s[threadIdx.x] = 0ull;
    __syncthreads();
    const u64 *rows = stat_rows(C);
    u64 sum = 0;
    for (uint32_t i = threadIdx.x; i < kStatRows * kStatCols; i += 1024) sum += rows[i];
    atomicAdd(&s[threadIdx.x % kStatCols], sum);
    __syncthreads();
    if (threadIdx.x < kWStats) (&C->relax)[threadIdx.x] += s[threadIdx.x];
}

// After a batch: its record for the host (`out`, unless null) and, if it is
// done, the counters for a next batch of rsz roots (none if 0).  Round 1's
// frontier is the batch's roots in order: root offset ro holds active-list
// slot ro and touched-list entry ro (k_w_init).
__global__ void k_w_close(WCounters *C, uint32_t rsz, WClosed *out)
{
    const uint32_t hold = C->hold;
    if (out) {
        out->rounds = C->rounds;
        out->held = hold;
        out->n_touched = C->n_touched;
    }
    if (hold || rsz == 0) return;
    C->n_act[0] = C->n_chunk[0] = C->n_chunk[1] = C->n_imp[0] = C->n_imp[1] = 0;
    C->a_top[0] = 0;
    C->n_act[1] = 1;
    C->a_top[1] = rsz;
    C->n_touched = rsz;
    C->need = C->need_bound = 0;
}

__global__ void k_w_unhold(WCounters *C) { C->hold = 0; }

// Earlier-batch labels of the batch roots -> root-distance table
// (roots_labels_buffer, WPARA:322-348, transposed): dcw[h][ro] = d(root
// rs + ro, hub h), indexed by hub id, and hmin[h] = the least of them.  Both
// are INF outside the batch roots' hubs (k_w_commit resets what was written).
// Lists are hub-sorted and every root holds the top-ranked hubs: walking them
// from the end staggers the roots' arrival at those hubs, so the plain read of
// hmin skips most atomics.  The root's list of `len` labels is walked by
// `parts` waves of which this is number `part`, two labels per lane and step.
__device__ inline void w_hub_fill(uint32_t ro, u64 base, uint32_t len, uint32_t part, uint32_t parts, WStore S,
                                  uint32_t *hmin, uint32_t *dcw)
{
    const uint32_t lane = lane_id();
    for (uint32_t k0 = part * 128; k0 < len; k0 += parts * 128) {
        u64 lab[2];
        uint32_t hm[2];
        bool ok[2];
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u) {
            const uint32_t k = k0 + 64 * u + lane;  // from the end
            ok[u] = k < len;
            lab[u] = ok[u] ? S.pool[base + (len - 1 - k)] : 0ull;
        }
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u) {
            const uint32_t h = (uint32_t)(lab[u] >> 32);
            if (ok[u]) {
                hm[u] = hmin[h];
                dcw[(uint64_t)h * kWB + ro] = (uint32_t)lab[u];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u)
            if (ok[u] && (uint32_t)lab[u] < hm[u]) atomicMin(&hmin[lab[u] >> 32], (uint32_t)lab[u]);
    }
}

// initialize_tables (WPARA:305-383): every root at distance 0 from itself,
// active with its own bit, and its earlier labels in the root-distance table.
// Four roots per block: the first four waves set the roots up, the other
// twelve (three per root) enter their labels, which nothing here changes.  One
// chunk reservation per block.
constexpr uint32_t kWInitFill = 3;
__global__ __launch_bounds__(256 * (1 + kWInitFill)) void k_w_init(uint32_t rs, uint32_t rsz, uint32_t gen_batch, const uint64_t *off,
                                                const uint32_t *adj, uint32_t *T, uint32_t *tmark, uint32_t *tlist,
                                                uint32_t *alist, u64 *ag, uint32_t *amask, uint32_t *aend, u64 *chunks,
                                                uint32_t *hmin, uint32_t *dcw, WStore S, WCounters *C)
{
    __shared__ uint32_t s_nch[4], s_c0;
    const uint32_t lane = lane_id(), wv = (threadIdx.x >> 6) & 3u, part = threadIdx.x >> 8;
    const uint32_t ro = blockIdx.x * 4 + wv;
    if (C->hold) return;
    if (part) {
        if (ro < rsz) w_hub_fill(ro, S.base[rs + ro], S.len[rs + ro], part - 1u, kWInitFill, S, hmin, dcw);
        __syncthreads();
        __syncthreads();
        return;
    }
    uint32_t nch = 0;
    if (ro < rsz) {
        const uint32_t r = rs + ro;
        if (lane == 0) {
            T[(uint64_t)r * kWB + ro] = 0;
            tmark[r] = gen_batch;
            tlist[ro] = r;
            alist[ro] = r;
            amask[ro] = 1u << (ro >> 6);
            const u64 nb = reserve_words(S.len[r], S.cap[r], rsz);
            if (nb) atomicAdd(&C->need_bound, nb);
        }
        if (lane < kWW) ag[(uint64_t)ro * kWW + lane] = (lane == (ro >> 6)) ? (1ull << (ro & 63)) : 0ull;
        const uint32_t pdeg = prefix_above(off, adj, r, rs);
        if (lane == 0) aend[ro] = pdeg;
        nch = (pdeg + kChunk - 1) / kChunk;
    }
    if (lane == 0) s_nch[wv] = nch;
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t tot = s_nch[0] + s_nch[1] + s_nch[2] + s_nch[3];
        s_c0 = tot ? atomicAdd(&C->n_chunk[1], tot) : 0u;
    }
    __syncthreads();
    uint32_t c0 = s_c0;
    for (uint32_t w = 0; w < wv; ++w) c0 += s_nch[w];
    for (uint32_t q = lane; q < nch; q += 64) chunks[c0 + q] = ((u64)(q * kChunk) << 32) | ro;
}


// Position of the rank-th set bit of m (rank < popcount(m)).
__device__ inline uint32_t w_nth_set_bit(u64 m, uint32_t rank)
{
    uint32_t pos = 0;
    uint32_t c = __popc((uint32_t)m);
    if (rank >= c) {
        rank -= c;
        m >>= 32;
        pos = 32;
    }
    uint32_t x = (uint32_t)m;
#pragma unroll
    for (uint32_t width = 16; width; width >>= 1) {
        c = __popc(x & ((1u << width) - 1u));
        if (rank >= c) {
            rank -= c;
            x >>= width;
            pos += width;
        }
    }
    return pos;
}

constexpr uint32_t kWPushWaves = 4;  // waves per k_w_push block
// Roots in a frontier word from which on k_w_push takes the word lane by lane,
// kWPushEdges edges at a time (weighted R-MAT 20: 612 ms without, 597 at 16,
// 598 at 24, 604 at 8; eight edges at a time 598).
constexpr uint32_t kWDense = 16, kWPushEdges = 4;

// Touched vertices up to which k_w_filter reads the roots' entries in place.
constexpr uint32_t kWDirectFilter = 4096;

constexpr uint32_t kWWitness = 2;  // witnesses k_w_filter takes at a time (1 and 4 measure the same)

// Batches in flight, from the kWAheadFrom-th on (weighted R-MAT 20: 2: 575
// ms, 1: 585, 3: 584, 4: 585, 7: 599 -- a batch that is held costs the empty
// launches of those behind it).
constexpr uint32_t kWAhead = 2, kWAheadFrom = 8;

// Rounds that a batch is enqueued with at most.  Batches differ: after one of
// 3,000 rounds the next ones of a path were given as many, at 7 us a round
// that does nothing (weighted path of 3,000 vertices: 108 ms, with 16 to 128:
// 38.3 to 39.9; 3,000 x 12 grid: 818 and 759-763; R-MAT 18: 86.5 either way).
constexpr uint32_t kWRoundsAhead = 32;

// Improved pairs of a tail up to which k_w_check reads single table entries.
constexpr uint32_t kWGather = 8;

// k_w_check reserves next-frontier slots per wave: kWAlistGrab active-list
// entries and up to kWChunkGrab push descriptors per atomic on the shared
// counters; a descriptor slot reserved but not used holds kWChunkPad (edge
// offset past every list), which k_w_push skips.
constexpr uint32_t kWAlistGrab = 64, kWChunkGrab = 64;
constexpr u64 kWChunkPad = 0xFFFFFFF0ull << 32;

// send_messages (WPARA:435-522): relax the frontier's edges toward tails
// ranked below each root.  A wave takes four 16-edge chunks (one edge per
// lane) and walks the root words of its edges' groups in step.  Chunks with
// many roots in a word go edge by edge, lane = root: the source's distances
// are read once for the chunk's edges, the tails' in whole lines.  For the
// others the (edge, root) relaxations of all 64 lanes are spread over the
// wave, 64 per step, so an edge with many roots does not hold up the others.
// The first batches' rounds, most of the time, are bound by the random lines
// of T that they read and update (about 2 TB/s).
__global__ __launch_bounds__(256) void k_w_push(uint32_t round, uint32_t rs, uint32_t rsz, uint32_t gen_batch,
                                                const uint64_t *off, const uint32_t *adj, const uint8_t *wgt,
                                                const uint32_t *alist, const u64 *ag, const uint32_t *amask,
                                                const uint32_t *aend, const u64 *chunks, uint32_t *T, u64 *I,
                                                uint32_t *tmark, uint32_t *tlist, u64 *imark, uint32_t *ilist,
                                                WStore S, WCounters *C)
{
    __shared__ u64 s_g[kWPushWaves][64], s_imp[kWPushWaves][64];
    __shared__ uint32_t s_ex[kWPushWaves][64], s_u[kWPushWaves][64], s_t[kWPushWaves][64], s_w[kWPushWaves][64];
    __shared__ uint32_t s_tl[kWPushWaves][64], s_il[kWPushWaves][64];  // entries on their way to the lists
    const uint32_t lane = lane_id(), wv = threadIdx.x >> 6;
    const uint32_t wave = blockIdx.x * kWPushWaves + wv;
    const uint32_t nwaves = gridDim.x * kWPushWaves;
    // Round `round` of the batch (slot round & 1; empty past the batch's
    // end).  Block 0 empties the other slot, which k_w_check fills.
    const uint32_t p = round & 1u;
    if (C->hold) return;
    const uint32_t nc = C->n_chunk[p];
    const u64 gen_round = ((u64)gen_batch << 24) | round;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (C->n_act[p]) C->rounds += 1;
        C->n_act[p ^ 1u] = 0;
        C->a_top[p ^ 1u] = 0;
        C->n_chunk[p ^ 1u] = 0;
    }
    uint32_t held_t = 0, held_i = 0;
    uint32_t n_relax = 0, n_imp = 0, n_bound = 0;  // (a list's reservation fits 32 bits, and a lane's few do)
    for (uint32_t c0 = wave * 4; c0 < nc; c0 += nwaves * 4) {
        const uint32_t c = c0 + (lane >> 4);
        uint32_t k = 0, u = 0, t = 0, w = 0, lim = 0, words = 0;
        const u64 desc = c < nc ? chunks[c] : kWChunkPad;
        if (desc != kWChunkPad) {
            k = (uint32_t)desc;
            const uint32_t e = (uint32_t)(desc >> 32) + (lane & (kChunk - 1));
            if (e < aend[k]) {
                u = alist[k];
                const uint64_t ei = off[u] + e;
                t = adj[ei];
                w = wgt[ei];
                lim = t - rs;  // roots with offset < lim rank above t
                words = amask[k] & (lim >= kWB ? ((1u << kWW) - 1u) : ((1u << ((lim + 63) / 64)) - 1u));
            }
        }
        s_u[wv][lane] = u;
        s_t[wv][lane] = t;
        s_w[wv][lane] = w;
        uint32_t wall = wave_or(words);
        bool got = false;
        while (wall) {
            const uint32_t wd = __ffs(wall) - 1;
            wall &= wall - 1;
            u64 g = 0, all = 0;
            if ((words >> wd) & 1u) {
                g = all = ag[(uint64_t)k * kWW + wd];
                if (lim < (wd + 1) * 64) g &= (1ull << (lim - wd * 64)) - 1ull;
            }
            // Chunks with many roots in this word: lane = root.
            u64 imp = 0;
            const u64 dense = __ballot(__popcll(all) >= (int)kWDense);
            for (u64 todo = dense; todo;) {
                const uint32_t l0 = (uint32_t)__ffsll(todo) - 1;
                u64 edges = todo & (0xFFFFull << (l0 & ~(kChunk - 1)));  // this chunk's
                todo &= ~edges;
                const u64 roots = readlane64(all, l0);
                const uint32_t *from = T + (uint64_t)__builtin_amdgcn_readlane(u, l0) * kWB + wd * 64;
                const uint32_t du = (roots >> lane) & 1ull ? from[lane] : kWInf;
                while (edges) {
                    uint32_t e[kWPushEdges], cur[kWPushEdges], cand[kWPushEdges], *to[kWPushEdges];
#pragma unroll
                    for (uint32_t j = 0; j < kWPushEdges; ++j) {
                        // (past the chunk's last edge: that edge again, relaxed by no lane)
                        const bool more = edges != 0ull;
                        e[j] = more ? (uint32_t)__ffsll(edges) - 1 : l0;
                        edges &= edges - 1;
                        const uint32_t le = more ? __builtin_amdgcn_readlane(lim, e[j]) : 0u;
                        to[j] = T + (uint64_t)__builtin_amdgcn_readlane(t, e[j]) * kWB + wd * 64;
                        const bool on = du != kWInf && wd * 64 + lane < le;
                        cand[j] = on ? du + __builtin_amdgcn_readlane(w, e[j]) : kWInf;
                        cur[j] = 0;
                        if (on) cur[j] = to[j][lane];
                        n_relax += on ? 1u : 0u;
                    }
#pragma unroll
                    for (uint32_t j = 0; j < kWPushEdges; ++j) {
                        bool better = false;
                        if (cand[j] < cur[j]) better = cand[j] < atomicMin(to[j] + lane, cand[j]);
                        const u64 who = __ballot(better);
                        if (lane == e[j]) imp |= who;
                    }
                }
            }
            if ((dense >> lane) & 1ull) g = 0;
            const uint32_t cnt = (uint32_t)__popcll(g);
            const uint32_t incl = wave_incl_scan(cnt);
            const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
            if (total) {
                s_g[wv][lane] = g;
                s_ex[wv][lane] = incl - cnt;
                s_imp[wv][lane] = 0ull;
                wave_lds_sync();
                for (uint32_t x0 = 0; x0 < total; x0 += 64) {
                    const uint32_t x = x0 + lane;
                    if (x >= total) continue;
                    uint32_t o = 0;
#pragma unroll
                    for (uint32_t sft = 32; sft; sft >>= 1)
                        if (s_ex[wv][o + sft] <= x) o += sft;
                    const uint32_t b = w_nth_set_bit(s_g[wv][o], x - s_ex[wv][o]);
                    const uint32_t ro = wd * 64 + b;
                    const uint32_t du = T[(uint64_t)s_u[wv][o] * kWB + ro];
                    if (du == kWInf) continue;
                    const uint32_t cand = du + s_w[wv][o];
                    ++n_relax;
                    // A plain read first: values only fall during the kernel, so
                    // one read as <= cand (even a stale one) makes the atomic a no-op.
                    uint32_t *tt = &T[(uint64_t)s_t[wv][o] * kWB + ro];
                    if (cand < *tt) {
                        const uint32_t old = atomicMin(tt, cand);
                        if (cand < old) atomicOr(&s_imp[wv][o], 1ull << b);
                    }
                }
                wave_lds_sync();
                imp |= s_imp[wv][lane];
            }
            if (imp) {
                atomicOr(&I[(uint64_t)t * kWW + wd], imp);
                got = true;
            }
            // The next word's writes must not overtake this word's reads.
            wave_lds_sync();
        }
        const bool new_t = got && tmark[t] != gen_batch && atomicExch(&tmark[t], gen_batch) != gen_batch;
        const bool new_i = got && imark[t] != gen_round && atomicExch(&imark[t], gen_round) != gen_round;
        list_append(&C->n_touched, tlist, s_tl[wv], held_t, new_t, t);
        if (new_t) n_bound += (uint32_t)reserve_words(S.len[t], S.cap[t], rsz);
        list_append(&C->n_imp[p], ilist, s_il[wv], held_i, new_i, t);
        n_imp += new_i ? 1u : 0u;
        // s_u / s_t / s_w are rewritten by the next step.
        wave_lds_sync();
    }
    list_flush(&C->n_touched, tlist, s_tl[wv], held_t);
    list_flush(&C->n_imp[p], ilist, s_il[wv], held_i);
    if (wave * 4 < nc) {
        const u64 t_bound = wave_total(n_bound & 0xFFFFu) + ((u64)wave_total(n_bound >> 16) << 16);
        if (lane == 0 && t_bound) atomicAdd(&C->need_bound, t_bound);
        add_stats<0>(stat_rows(C), wave, {n_relax, n_imp});
    }
}

// distance_query's first loop (WPARA:569-580) for every improved pair of an
// improved tail: one wave per tail, lane l owns roots 8l..8l+7.  Pruned pairs
// stop propagating; the others become the tail's next frontier bitmap.
// Bound by instruction issue where a batch is large (4.1 G of them, 6.7 of
// 9.8 ms, in the largest round of weighted R-MAT 20; the hubs' rows come from
// L2): the sums through the hubs are kept as a saturated minimum per pair, two
// instructions per hub where comparing each took seven (build 550 -> 504 ms).
__global__ __launch_bounds__(256) void k_w_check(uint32_t round, uint32_t rs, const uint32_t *ilist, const uint64_t *off,
                                                 const uint32_t *adj, uint32_t *T, u64 *I, u64 *P, WStore S,
                                                 const uint32_t *hmin, const uint32_t *dcw,
                                                 uint32_t *alist, u64 *ag, uint32_t *amask, uint32_t *aend,
                                                 u64 *chunks, WCounters *C)
{
    const uint32_t lane = lane_id();
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    const uint32_t p = round & 1u;
    if (C->hold) return;
    const uint32_t nimp = C->n_imp[p];
    if (blockIdx.x == 0 && threadIdx.x == 0) C->n_imp[p ^ 1u] = 0;
    uint32_t n_pruned = 0;
    uint32_t a_next = 0, a_left = 0, c_next = 0, c_left = 0, my_act = 0;
    for (uint32_t i = wave; i < nimp; i += nwaves) {
        const uint32_t t = ilist[i];
        uint8_t *Ib = reinterpret_cast<uint8_t *>(I + (uint64_t)t * kWW);
        uint8_t *Pb = reinterpret_cast<uint8_t *>(P + (uint64_t)t * kWW);
        const uint32_t imp = Ib[lane];
        // Clear after every lane has read (the store depends on the ballot).
        if (__ballot(imp != 0) != 0ull) Ib[lane] = 0;
        uint32_t maxd = 0;
        uint4 t0 = make_uint4(0, 0, 0, 0), t1 = t0;
        if (imp) {
            const uint4 *row = reinterpret_cast<const uint4 *>(T + (uint64_t)t * kWB + lane * 8);
            t0 = row[0];
            t1 = row[1];
        }
        // Tentative distances of the improved pairs, 0 for the others: a sum
        // through an earlier hub is at least 2.
        uint32_t dv[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            dv[q] = (imp >> q) & 1u ? dv[q] : 0u;
            maxd = max(maxd, dv[q]);
        }
        const uint32_t wmax = wave_max(maxd);
        uint32_t prune = 0;
        const uint32_t len = uniform32(S.len[t]);
        const u64 base = uniform64(S.base[t]);
        // Row phase: while more than kWGather improved pairs are unpruned,
        // lanes hold roots (8 each) and read the passing hubs' row slices.
        // The first hubs usually prune most pairs; once a 4-hub group leaves
        // at most kWGather unpruned, the labels not yet read go to the gather
        // phase.
        uint32_t j_gather = 0;
        if (wave_total(__popc(imp)) > kWGather) {
            j_gather = len;
            uint32_t best[8];  // the least sums through the hubs so far
#pragma unroll
            for (int q = 0; q < 8; ++q) best[q] = kWInf;
            for (uint32_t j0 = 0; j0 < len; j0 += 64) {
                const uint32_t j = j0 + lane;
                uint32_t h = 0, d = kWInf;
                if (j < len) {
                    const u64 lab = S.pool[base + j];
                    h = (uint32_t)(lab >> 32);
                    d = (uint32_t)lab;
                }
                // hmin is INF for hubs no batch root holds
                const bool pass = j < len && __builtin_elementwise_add_sat(d, hmin[h]) <= wmax;
                u64 m = __ballot(pass);
                // Up to four passing hubs per step: their row loads go out
                // together (32 B per lane each), and only lanes that still hold an
                // unpruned improved pair load.
                bool few = false;
                while (m) {
                    // (past the last one: that one again)
                    uint32_t src[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        src[u] = m ? (uint32_t)__ffsll(m) - 1 : src[u ? u - 1 : 0];
                        m &= m - 1;
                    }
                    if (imp & ~prune) {
                        uint4 r0[4], r1[4];
                        uint32_t dd[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            dd[u] = __builtin_amdgcn_readlane(d, src[u]);
                            const uint32_t *hub = dcw + (uint64_t)__builtin_amdgcn_readlane(h, src[u]) * kWB;
                            r0[u] = reinterpret_cast<const uint4 *>(hub)[lane * 2];
                            r1[u] = reinterpret_cast<const uint4 *>(hub)[lane * 2 + 1];
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint32_t x[8] = {r0[u].x, r0[u].y, r0[u].z, r0[u].w, r1[u].x, r1[u].y, r1[u].z, r1[u].w};
#pragma unroll
                            for (int q = 0; q < 8; ++q)
                                best[q] = min(best[q], __builtin_elementwise_add_sat(x[q], dd[u]));
                        }
#pragma unroll
                        for (int q = 0; q < 8; ++q) prune |= best[q] <= dv[q] ? 1u << q : 0u;
                    }
                    if (wave_total(__popc(imp & ~prune)) <= kWGather) {
                        few = true;
                        break;
                    }
                }
                if (few) {
                    // the step's passing hubs not yet read start the gather phase
                    const uint32_t nxt = m ? j0 + (uint32_t)__ffsll(m) - 1 : j0 + 64;
                    j_gather = nxt < len ? nxt : len;
                    break;
                }
            }
        }
        // Gather phase: the (at most kWGather) improved pairs still unpruned
        // are checked hub-parallel over labels j_gather.. : lanes hold labels
        // and read one table entry per pair, 128 labels per step with the
        // next step's labels loaded while this one runs.  croot / cdv: the
        // pairs' root offsets and tentative distances (wave-uniform); cpr:
        // which are pruned.
        uint32_t croot[kWGather], cdv[kWGather];
        uint32_t ncand_t = 0, cpr = 0;
        {
            uint32_t rest = imp & ~prune;
#pragma unroll
            for (uint32_t k = 0; k < kWGather; ++k) {
                const unsigned long long m = __ballot(rest != 0u);
                croot[k] = 0u;
                cdv[k] = 0u;
                if (m) {
                    const uint32_t l0 = (uint32_t)__ffsll(m) - 1;
                    const uint32_t bits = uniform32(__shfl(rest, (int)l0));
                    const uint32_t q = (uint32_t)__ffs(bits) - 1;
                    // dv[q] of lane l0 (unrolled select: no runtime index into dv)
                    uint32_t myd = 0;
#pragma unroll
                    for (uint32_t qq = 0; qq < 8; ++qq)
                        if (qq == q) myd = dv[qq];
                    croot[k] = 8 * l0 + q;
                    cdv[k] = uniform32(__shfl(myd, (int)l0));
                    if (lane == l0) rest &= rest - 1;
                    ++ncand_t;
                }
            }
        }
        if (ncand_t && j_gather < len) {
            auto gather_pass = [&](uint32_t d, uint32_t h, uint32_t hm) {
                uint32_t x[kWGather];
                const uint32_t least = __builtin_elementwise_add_sat(d, hm);
                const uint32_t *row = dcw + (uint64_t)h * kWB;
#pragma unroll
                for (uint32_t k = 0; k < kWGather; ++k) {
                    x[k] = kWInf;
                    if (k < ncand_t && !((cpr >> k) & 1u) && least <= cdv[k]) x[k] = row[croot[k]];
                }
                // (a tentative distance is below INF)
#pragma unroll
                for (uint32_t k = 0; k < kWGather; ++k)
                    if (__ballot(__builtin_elementwise_add_sat(d, x[k]) <= cdv[k]) != 0ull) cpr |= 1u << k;
            };
            const u64 gb = base + j_gather;
            const uint32_t glen = len - j_gather;
            u64 la = lane < glen ? S.pool[gb + lane] : 0ull, lb = lane + 64 < glen ? S.pool[gb + lane + 64] : 0ull;
            for (uint32_t j0 = 0; j0 < glen; j0 += 128) {
                const uint32_t ja = j0 + lane, jb = j0 + 64 + lane;
                const u64 ca = la, cbl = lb;
                la = ja + 128 < glen ? S.pool[gb + ja + 128] : 0ull;
                lb = jb + 128 < glen ? S.pool[gb + jb + 128] : 0ull;
                // (past the list: d = hmin = INF, so nothing is read)
                uint32_t da = kWInf, db = kWInf, sa = 0, sb = 0, ma = kWInf, mb = kWInf;
                if (ja < glen) {
                    sa = (uint32_t)(ca >> 32);
                    da = (uint32_t)ca;
                    ma = hmin[sa];
                }
                if (jb < glen) {
                    sb = (uint32_t)(cbl >> 32);
                    db = (uint32_t)cbl;
                    mb = hmin[sb];
                }
                gather_pass(da, sa, ma);
                gather_pass(db, sb, mb);
                if (cpr == (1u << ncand_t) - 1u) break;
            }
#pragma unroll
            for (uint32_t k = 0; k < kWGather; ++k)
                if (((cpr >> k) & 1u) && lane == (croot[k] >> 3)) prune |= 1u << (croot[k] & 7u);
        }
        const uint32_t live = imp & ~prune;
        n_pruned += __popc(imp & prune);
        // pruned-at-current-value bits: set for pruned, cleared for live
        if (imp) Pb[lane] = (uint8_t)((Pb[lane] & ~imp) | (imp & prune));
        const u64 any = __ballot(live != 0);
        if (!any) continue;
        // Next-frontier slots come from per-wave reservations, capped by the
        // tails this wave has left in the launch (grid-stride).
        const uint32_t rem = (nimp - 1 - i) / nwaves + 1;
        if (a_left == 0) {
            const uint32_t grab = rem < kWAlistGrab ? rem : kWAlistGrab;
            uint32_t b0 = 0;
            if (lane == 0) b0 = atomicAdd(&C->a_top[p ^ 1u], grab);
            a_next = __shfl(b0, 0);
            a_left = grab;
        }
        const uint32_t k = a_next++;
        --a_left;
        ++my_act;
        reinterpret_cast<uint8_t *>(ag + (uint64_t)k * kWW)[lane] = (uint8_t)live;
        uint32_t wmask = 0;
#pragma unroll
        for (int w = 0; w < (int)kWW; ++w)
            if ((any >> (8 * w)) & 0xFFull) wmask |= 1u << w;
        const uint32_t pdeg = prefix_above(off, adj, t, rs);
        if (lane == 0) {
            alist[k] = t;
            amask[k] = wmask;
            aend[k] = pdeg;
        }
        const uint32_t nch = (pdeg + kChunk - 1) / kChunk;
        if (nch > c_left) {
            for (uint32_t q = lane; q < c_left; q += 64) chunks[c_next + q] = kWChunkPad;
            const uint64_t guess = (uint64_t)nch * rem;  // descriptors left if t is typical
            const uint32_t cap = guess < kWChunkGrab ? (uint32_t)guess : kWChunkGrab;
            const uint32_t want = nch > cap ? nch : cap;
            uint32_t b0 = 0;
            if (lane == 0) b0 = atomicAdd(&C->n_chunk[p ^ 1u], want);
            c_next = __shfl(b0, 0);
            c_left = want;
        }
        for (uint32_t q = lane; q < nch; q += 64) chunks[c_next + q] = ((u64)(q * kChunk) << 32) | k;
        c_next += nch;
        c_left -= nch;
    }
    for (uint32_t q = lane; q < c_left; q += 64) chunks[c_next + q] = kWChunkPad;
    if (lane == 0 && my_act) C->n_act[p ^ 1u] = 1u;  // (every writer writes the same)
    if (wave < nimp) add_stats<2>(stat_rows(C), wave, {n_pruned});
}

// The batch roots' mutual entries, transposed for the filter: RT[h][r] =
// T[rs + r][h] and bit r of PT[h] = pruned bit h of root rs + r, so a witness
// h's column reads as one contiguous row.  One block per 64 x 64 tile (four
// waves, sixteen rows each); roots past the batch read as INF / unpruned.
__global__ __launch_bounds__(256) void k_w_roots_t(uint32_t rs, uint32_t rsz, const uint32_t *T, const u64 *P,
                                                   uint32_t *RT, u64 *PT)
{
    __shared__ uint32_t tile[64][65];
    const uint32_t lane = lane_id(), wv = threadIdx.x >> 6;
    const uint32_t r0 = (blockIdx.x % (kWB / 64)) * 64, h0 = (blockIdx.x / (kWB / 64)) * 64;
    for (uint32_t i = wv; i < 64; i += 4) {
        const uint32_t r = r0 + i;
        tile[i][lane] = r < rsz ? T[(uint64_t)(rs + r) * kWB + h0 + lane] : kWInf;
    }
    __syncthreads();
    for (uint32_t j = wv; j < 64; j += 4) RT[(uint64_t)(h0 + j) * kWB + r0 + lane] = tile[lane][j];
    // Pruned bits: lane = root r0 + lane, ballot over the roots per witness.
    if (wv == 0) {
        const uint32_t r = r0 + lane;
        const u64 pw = r < rsz ? P[(uint64_t)(rs + r) * kWW + h0 / 64] : 0ull;
        u64 mine = 0;
        for (uint32_t h = 0; h < 64; ++h) {
            const u64 bits = __ballot((pw >> h) & 1ull);
            if (lane == h) mine = bits;
        }
        PT[(uint64_t)(h0 + lane) * kWW + r0 / 64] = mine;
    }
}

// filter_out_labels (WPARA:1100-1228): one wave per touched vertex; surviving
// pairs (finite, not pruned) are dropped if an earlier batch root h witnesses
// S(v,h) + S(r,h) <= S(v,r).  The witnesses go through LDS, and a lane reads
// of a witness's row only while it has a pair left that it could drop (650 K
// vertices, 128 roots: 15.1 -> 9.8 ms).  Reads T/P only, so every wave sees the same
// pre-filter state; the kept bitmap goes to I and the pool words the commit
// may reserve are summed into C->need.  kDirect: the roots' entries come from
// T/P rows directly (8 scattered reads per witness and lane, no transpose
// kernel; for batches that touch few vertices), else from RT/PT.
// A batch enqueued in one go (gate) is held here if its rounds have not ended
// (`slot`: where the next frontier would be) or if its commit might not fit
// the pool: then this kernel and all later ones do nothing until the host has
// seen to it.
template <bool kDirect>
__global__ __launch_bounds__(256) void k_w_filter(uint32_t rs, uint32_t rsz, const uint32_t *tlist,
                                                  const uint32_t *T, const u64 *P, const uint32_t *RT, const u64 *PT,
                                                  u64 *I, WStore S, WCounters *C, uint32_t gate, uint32_t slot)
{
    // (every block decides alike: nothing here changes what it reads)
    if (gate) {
        if (C->hold) return;
        if (C->n_act[slot] != 0 || C->pool_top + C->need_bound > S.pool_size) {
            if (blockIdx.x == 0 && threadIdx.x == 0) C->hold = 1;
            return;
        }
    }
    __shared__ uint2 s_wit[4][kWB];
    const uint32_t lane = lane_id();
    const uint32_t wib = threadIdx.x >> 6;
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    const uint32_t nt = C->n_touched;
    __shared__ u64 s_lab, s_need;
    if (threadIdx.x == 0) s_lab = s_need = 0ull;
    __syncthreads();
    uint32_t n_filt = 0;
    u64 n_lab = 0, n_need = 0;
    for (uint32_t i = wave; i < nt; i += nwaves) {
        const uint32_t v = tlist[i];
        const uint8_t pb = reinterpret_cast<const uint8_t *>(P + (uint64_t)v * kWW)[lane];
        uint32_t dv[8];
        uint32_t surv = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            dv[q] = T[(uint64_t)v * kWB + lane * 8 + q];
            if (dv[q] != kWInf && !((pb >> q) & 1u)) surv |= 1u << q;
        }
        // The vertex's surviving pairs, roots ascending: the witnesses.
        const uint32_t cnt = __popc(surv);
        const uint32_t incl = wave_incl_scan(cnt);
        const uint32_t nwit = __builtin_amdgcn_readlane(incl, 63);
        {
            uint32_t at = incl - cnt;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if ((surv >> q) & 1u) s_wit[wib][at++] = make_uint2(lane * 8 + q, dv[q]);
        }
        wave_lds_sync();
        uint32_t drop = 0;
        for (uint32_t w = 0; w < nwit; w += kWWitness) {
            // Column h of the roots' entries for kWWitness witnesses h, 8 consecutive
            // roots per lane; only lanes that hold a root ranked below h and not
            // yet dropped read.
            uint32_t h[kWWitness], dvh[kWWitness], todo[kWWitness], drh[kWWitness][8], prh[kWWitness];
#pragma unroll
            for (uint32_t u = 0; u < kWWitness; ++u) {
                const uint2 x = s_wit[wib][min(w + u, nwit - 1)];
                h[u] = x.x;
                dvh[u] = x.y;
                const uint32_t below = lane * 8 > h[u] ? 0xFFu : lane * 8 + 7 <= h[u] ? 0u : 0xFFu & (0xFEu << (h[u] - lane * 8));
                todo[u] = surv & ~drop & below;
                prh[u] = 0;
#pragma unroll
                for (int q = 0; q < 8; ++q) drh[u][q] = kWInf;
                if (!todo[u]) continue;
                if constexpr (kDirect) {
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        const uint32_t ro = lane * 8 + q;
                        if ((todo[u] >> q) & 1u) {
                            drh[u][q] = T[(uint64_t)(rs + ro) * kWB + h[u]];
                            prh[u] |= (uint32_t)((P[(uint64_t)(rs + ro) * kWW + h[u] / 64] >> (h[u] % 64)) & 1ull) << q;
                        }
                    }
                } else {
                    const uint4 *rt = reinterpret_cast<const uint4 *>(RT + (uint64_t)h[u] * kWB + lane * 8);
                    const uint4 ra = rt[0], rb = rt[1];
                    drh[u][0] = ra.x, drh[u][1] = ra.y, drh[u][2] = ra.z, drh[u][3] = ra.w;
                    drh[u][4] = rb.x, drh[u][5] = rb.y, drh[u][6] = rb.z, drh[u][7] = rb.w;
                    prh[u] = reinterpret_cast<const uint8_t *>(PT + (uint64_t)h[u] * kWW)[lane];
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < kWWitness; ++u) {
                uint32_t by = 0;  // (a surviving pair's distance is below INF)
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    by |= __builtin_elementwise_add_sat(drh[u][q], dvh[u]) <= dv[q] ? 1u << q : 0u;
                drop |= by & todo[u] & ~prh[u];
            }
        }
        // (the next vertex's list must not overtake these reads)
        wave_lds_sync();
        const uint32_t keep = surv & ~drop;
        n_filt += __popc(drop);
        // The improved bitmap is all zero once the rounds end; it carries the
        // kept pairs to the commit kernel.
        reinterpret_cast<uint8_t *>(I + (uint64_t)v * kWW)[lane] = (uint8_t)keep;
        const uint32_t total = wave_total(__popc(keep));
        if (!total) continue;
        n_lab += total;
        if (lane == 0) n_need += reserve_words(S.len[v], S.cap[v], total);
    }
    if (wave < nt) add_stats<3>(stat_rows(C), wave, {n_filt});
    if (lane == 0) {
        if (n_lab) atomicAdd(&s_lab, n_lab);
        if (n_need) atomicAdd(&s_need, n_need);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_lab) atomicAdd(&C->labels, s_lab);
        if (s_need) atomicAdd(&C->need, s_need);
    }
}

// update_index (WPARA:961-990) and reset_tables (WPARA:918-956) in one pass
// over the touched vertices: a wave appends a vertex's kept pairs, hubs
// ascending (batches are committed in root order and each lane's roots follow
// the lower lanes'), clears the carried bitmap and empties its T / P rows; the
// batch roots (touched-list entries 0..rsz-1) first clear the root-distance
// entries their labels wrote.  Waves take up to 64 vertices at a time and the
// pool words for them with one atomic: one per vertex, all on one word, was
// most of a large batch's commit (650 K vertices: 7.7 ms, now 0.9).
__global__ __launch_bounds__(256) void k_w_commit(uint32_t rs, uint32_t rsz, const uint32_t *tlist, uint32_t *T, u64 *P,
                                                  u64 *I, uint32_t *hmin, uint32_t *dcw, WStore S, WCounters *C)
{
    if (C->hold) return;
    const uint32_t lane = lane_id();
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    const uint32_t nt = C->n_touched;
    const uint32_t group = min(64u, max(1u, nt / nwaves));
    for (uint32_t i0 = wave * group; i0 < nt; i0 += nwaves * group) {
        const uint32_t m = min(group, nt - i0);
        // Lane i: the group's i-th vertex, its list and the words it moves to.
        uint32_t v = 0, total = 0, len = 0, need = 0;
        u64 base = 0;
        if (lane < m) {
            v = tlist[i0 + lane];
            const ulonglong2 *kept = reinterpret_cast<const ulonglong2 *>(I + (uint64_t)v * kWW);
#pragma unroll
            for (uint32_t x = 0; x < kWW / 2; ++x) total += (uint32_t)(__popcll(kept[x].x) + __popcll(kept[x].y));
            len = S.len[v];
            base = S.base[v];
            if (total) need = (uint32_t)reserve_words(len, S.cap[v], total);
        }
        const uint32_t incl = wave_incl_scan(need);
        const uint32_t words = __builtin_amdgcn_readlane(incl, 63);
        u64 nb = 0;
        if (words) {
            if (lane == 0) nb = atomicAdd(&C->pool_top, (u64)words);
            nb = uniform64(nb);
        }
        const bool fits = words == 0 || nb + words <= S.pool_size;
        if (!fits && lane == 0) atomicOr(&C->overflow, 1u);
        const u64 to = need ? nb + (incl - need) : base;
        if (lane < m && total && fits) {
            S.len[v] = len + total;
            if (need) {
                S.base[v] = to;
                S.cap[v] = need;
            }
        }
        for (uint32_t s = 0; s < m; ++s) {
            const uint32_t vs = __builtin_amdgcn_readlane(v, s), ls = __builtin_amdgcn_readlane(len, s);
            const u64 from = readlane64(base, s);
            if (i0 + s < rsz) {
                // root offset i0 + s: its labels are those k_w_init entered
                for (uint32_t j = lane; j < ls; j += 64) {
                    const uint32_t h = (uint32_t)(S.pool[from + j] >> 32);
                    dcw[(uint64_t)h * kWB + i0 + s] = kWInf;
                    hmin[h] = kWInf;
                }
            }
            uint4 *row = reinterpret_cast<uint4 *>(T + (uint64_t)vs * kWB + lane * 8);
            if (__builtin_amdgcn_readlane(total, s)) {
                uint8_t *Kb = reinterpret_cast<uint8_t *>(I + (uint64_t)vs * kWW);
                const uint32_t keep = Kb[lane];
                uint4 r0 = make_uint4(0, 0, 0, 0), r1 = r0;
                if (keep) {
                    r0 = row[0];
                    r1 = row[1];
                    Kb[lane] = 0;
                }
                const u64 dst = readlane64(to, s);
                if (__builtin_amdgcn_readlane(need, s) && fits)
                    for (uint32_t j = lane; j < ls; j += 64) S.pool[dst + j] = S.pool[from + j];
                const uint32_t cnt = __popc(keep);
                u64 at = dst + ls + wave_incl_scan(cnt) - cnt;
                const uint32_t d[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
                for (uint32_t q = 0; q < 8; ++q)
                    if (fits && ((keep >> q) & 1u)) S.pool[at++] = ((u64)(rs + lane * 8 + q) << 32) | d[q];
            }
            // The row goes back to INF.
            row[0] = row[1] = make_uint4(kWInf, kWInf, kWInf, kWInf);
            if (lane < kWW) P[(uint64_t)vs * kWW + lane] = 0ull;
        }
    }
}

__global__ void k_w_fill(uint32_t *p, uint64_t count, uint32_t val)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) p[i] = val;
}

__global__ void k_w_zero64(u64 *p, uint64_t count)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) p[i] = 0ull;
}

// Copies list v (len[v] words at pool[base[v]]) to dst[dst_off[v]].
__global__ __launch_bounds__(256) void k_w_move(uint32_t n, const u64 *pool, const u64 *base, const uint32_t *len,
                                                const uint64_t *dst_off, u64 *dst)
{
    const uint32_t lane = lane_id();
    const uint32_t nw = (gridDim.x * blockDim.x) >> 6;
    for (uint32_t v = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; v < n; v += nw) {
        const uint64_t o = dst_off[v], b = base[v];
        const uint32_t L = len[v];
        for (uint32_t j = lane; j < L; j += 64) dst[o + j] = pool[b + j];
    }
}

__global__ void k_w_split(uint64_t total, const u64 *lab, uint32_t *hub, uint32_t *dist)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        hub[i] = (uint32_t)(lab[i] >> 32);
        dist[i] = (uint32_t)lab[i];
    }
}

}  // namespace

pado_gpu_status build_weighted(pado_gpu_graph *g, pado_gpu_index *idx, uint32_t batch_req)
{
    hipStream_t st = g->ctx->stream;
    const uint32_t n = g->n;
    const uint32_t batch = (batch_req == 0 || batch_req > kWB) ? kWB : batch_req;
    DevBuf<uint32_t> T, tmark, tlist, ilist, alist, amask, aend, hmin, dcw, len, cap;
    DevBuf<u64> P, I, ag, chunks, pool, base, imark;
    DevBuf<uint32_t> RT;  // batch roots' entries, transposed for the filter
    DevBuf<u64> PT;
    DevBuf<WCounters> ctr;
    WorkPool *wp = g->work.get();
    PADO_TRY(T.alloc((uint64_t)n * kWB, wp));
    PADO_TRY(RT.alloc((uint64_t)kWB * kWB, wp));
    PADO_TRY(PT.alloc((uint64_t)kWB * kWW, wp));
    PADO_TRY(P.alloc((uint64_t)n * kWW, wp));
    PADO_TRY(I.alloc((uint64_t)n * kWW, wp));
    // Per-wave reservations in k_w_check leave holes: up to kWAlistGrab
    // active-list slots per wave beyond the real ones, and padded
    // descriptors fewer than the real ones plus kWChunkGrab per wave.
    const uint64_t check_waves = 4ull * kAddGrid;
    const uint64_t alist_cap = (uint64_t)n + kWAlistGrab * check_waves;
    PADO_TRY(ag.alloc(alist_cap * kWW, wp));
    PADO_TRY(chunks.alloc(2 * (g->m / kChunk + (uint64_t)n) + kWChunkGrab * check_waves + 64, wp));
    PADO_TRY(tmark.alloc(n, wp));
    PADO_TRY(tlist.alloc(n, wp));
    PADO_TRY(imark.alloc(n, wp));
    PADO_TRY(ilist.alloc(n, wp));
    PADO_TRY(alist.alloc(alist_cap, wp));
    PADO_TRY(amask.alloc(alist_cap, wp));
    PADO_TRY(aend.alloc(alist_cap, wp));
    PADO_TRY(hmin.alloc(n, wp));
    PADO_TRY(len.alloc(n, wp));
    PADO_TRY(cap.alloc(n, wp));
    PADO_TRY(base.alloc(n, wp));
    PADO_TRY(ctr.alloc(1 + (kStatRows * kStatCols * 8 + sizeof(WCounters) - 1) / sizeof(WCounters), wp));
    u64 pool_size = std::max<u64>(1ull << 22, 32ull * n);
    PADO_TRY(pool.alloc(pool_size, wp));
    uint32_t dc_slots = std::min<uint32_t>(n, 1u << 14);
    PADO_TRY(dcw.alloc((uint64_t)dc_slots * kWB, wp));
    const uint32_t fg = 4096;
    hipLaunchKernelGGL(k_w_fill, dim3(fg), dim3(256), 0, st, dcw.p, (uint64_t)dc_slots * kWB, kWInf);
    hipLaunchKernelGGL(k_w_fill, dim3(fg), dim3(256), 0, st, T.p, (uint64_t)n * kWB, kWInf);
    hipLaunchKernelGGL(k_w_zero64, dim3(fg), dim3(256), 0, st, P.p, (uint64_t)n * kWW);
    hipLaunchKernelGGL(k_w_zero64, dim3(fg), dim3(256), 0, st, I.p, (uint64_t)n * kWW);
    hipLaunchKernelGGL(k_w_fill, dim3(fg), dim3(256), 0, st, tmark.p, (uint64_t)n, 0u);
    hipLaunchKernelGGL(k_w_zero64, dim3(fg), dim3(256), 0, st, imark.p, (uint64_t)n);
    hipLaunchKernelGGL(k_w_fill, dim3(fg), dim3(256), 0, st, hmin.p, (uint64_t)n, kWInf);
    hipLaunchKernelGGL(k_w_fill, dim3(fg), dim3(256), 0, st, len.p, (uint64_t)n, 0u);
    hipLaunchKernelGGL(k_w_fill, dim3(fg), dim3(256), 0, st, cap.p, (uint64_t)n, 0u);
    hipLaunchKernelGGL(k_w_zero64, dim3(fg), dim3(256), 0, st, base.p, (uint64_t)n);
    PADO_HIP(hipMemsetAsync(ctr.p, 0, ctr.n * sizeof(WCounters), st));
    PinnedBuf<WHost> pin;
    PADO_TRY(pin.alloc(wp, st));
    std::memset(pin.p, 0, sizeof(WHost));
    WCounters *h = &pin.p->c;
    volatile WClosed *ring = pin.p->ring;
    void *ring_dev = nullptr;
    PADO_HIP(hipHostGetDevicePointer(&ring_dev, pin.p->ring, 0));
    hipEvent_t ev[kWRing] = {};
    struct EventFree {
        hipEvent_t *e;
        ~EventFree()
        {
            for (uint32_t i = 0; i < kWRing; ++i)
                if (e[i]) (void)hipEventDestroy(e[i]);
        }
    } evf{ev};
    for (hipEvent_t &e : ev) PADO_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));

    WStore S{pool.p, base.p, len.p, cap.p, pool_size};
    // The first batch takes an eighth of the roots (one word of them, of 512):
    // nothing prunes its searches, and its labels prune the next batch's.
    // Any split of the rank order into batches yields the same label set.
    // Weighted R-MAT 20: a quarter 503 ms, an eighth 491, a sixteenth 499, a
    // 32nd 503; growing by doubling from either 498 to 511.
    const uint32_t first = std::min(n, std::max<uint32_t>(1u, batch / 8));
    const uint32_t nb = 1 + (n - first + batch - 1) / batch;
    auto roots_start = [&](uint32_t b) { return b ? first + (b - 1) * batch : 0u; };
    auto roots_size = [&](uint32_t b) { return b >= nb ? 0u : std::min(b ? batch : first, n - roots_start(b)); };
    auto rounds = [&](uint32_t b, uint32_t done, uint32_t more) {
        const uint32_t rs = roots_start(b), rsz = roots_size(b), gen_batch = b + 1;
        for (uint32_t round = done + 1; round <= done + more; ++round) {
            hipLaunchKernelGGL(k_w_push, dim3(kPushGrid), dim3(256), 0, st, round, rs, rsz, gen_batch, g->off.p,
                               g->adj.p, g->w.p, alist.p, ag.p, amask.p, aend.p, chunks.p, T.p, I.p, tmark.p,
                               tlist.p, imark.p, ilist.p, S, ctr.p);
            hipLaunchKernelGGL(k_w_check, dim3(kAddGrid), dim3(256), 0, st, round, rs, ilist.p, g->off.p, g->adj.p,
                               T.p, I.p, P.p, S, hmin.p, dcw.p, alist.p, ag.p, amask.p, aend.p,
                               chunks.p, ctr.p);
        }
    };
    // Blocks for the touched vertices, by how many the last batch had.
    auto touched_grid = [](uint32_t touched) { return std::min<uint32_t>(2048u, std::max<uint32_t>(256u, touched / 2)); };
    // Few touched vertices: the filter reads the roots' entries in place
    // instead of transposing them first.
    auto filter = [&](uint32_t b, uint32_t touched, uint32_t gate, uint32_t slot) {
        const uint32_t rs = roots_start(b), rsz = roots_size(b);
        const dim3 grid(touched_grid(touched));
        if (touched <= kWDirectFilter) {
            hipLaunchKernelGGL(k_w_filter<true>, grid, dim3(256), 0, st, rs, rsz, tlist.p, T.p, P.p, RT.p, PT.p, I.p,
                               S, ctr.p, gate, slot);
        } else {
            hipLaunchKernelGGL(k_w_roots_t, dim3((kWB / 64) * (kWB / 64)), dim3(256), 0, st, rs, rsz, T.p, P.p, RT.p,
                               PT.p);
            hipLaunchKernelGGL(k_w_filter<false>, grid, dim3(256), 0, st, rs, rsz, tlist.p, T.p, P.p, RT.p, PT.p, I.p,
                               S, ctr.p, gate, slot);
        }
    };
    auto commit = [&](uint32_t b, uint32_t touched) {
        const uint32_t rs = roots_start(b), rsz = roots_size(b);
        hipLaunchKernelGGL(k_w_commit, dim3(touched_grid(touched)), dim3(256), 0, st, rs, rsz, tlist.p, T.p, P.p, I.p,
                           hmin.p, dcw.p, S, ctr.p);
        hipLaunchKernelGGL(k_w_close, dim3(1), dim3(1), 0, st, ctr.p, roots_size(b + 1),
                           static_cast<WClosed *>(ring_dev) + b % kWRing);
    };
    // Batches are enqueued whole, with as many rounds as the last three needed
    // at most (up to kWRoundsAhead), and one ahead of the host's look at their
    // records, so that the later ones (38 us of kernels each) do not wait for
    // the host between their rounds and their filter.  A batch whose rounds
    // turn out not to have ended, or whose labels might not fit the pool,
    // holds everything behind it (k_w_filter); the host then ends it step by
    // step and goes on from there.  Weighted R-MAT 20: 597 -> 576 ms; 200 K
    // vertices: 80 -> 75.
    constexpr uint32_t kRoundHistory = 3;
    uint32_t hist[kRoundHistory] = {}, launched[kWRing] = {};
    hist[0] = 6;
    uint32_t next = 0, touched = n;  // batches enqueued; vertices the last batch touched
    u64 rounds_seen = 0;
    hipLaunchKernelGGL(k_w_close, dim3(1), dim3(1), 0, st, ctr.p, roots_size(0), (WClosed *)nullptr);
    for (uint32_t b = 0; b < nb; ++b) {
        // (the first few differ too much from each other to go ahead)
        const uint32_t ahead = b < kWAheadFrom ? 1u : kWAhead;
        for (; next < nb && next < b + ahead; ++next) {
            const uint32_t rs = roots_start(next), rsz = roots_size(next);
            // The hubs of the batch roots' labels are ids below the batch end, so
            // that many table rows always suffice (no device round trip).  A
            // batch that is held needs the table its rounds began with.
            if (rs + rsz > dc_slots) {
                if (next > b) break;
                dc_slots = std::min<uint32_t>(n, std::max<uint32_t>(rs + rsz, dc_slots * 2));
                PADO_TRY(dcw.alloc((uint64_t)dc_slots * kWB, wp));
                hipLaunchKernelGGL(k_w_fill, dim3(fg), dim3(256), 0, st, dcw.p, (uint64_t)dc_slots * kWB, kWInf);
            }
            hipLaunchKernelGGL(k_w_init, dim3((rsz * 64 + 255) / 256), dim3(256 * (1 + kWInitFill)), 0, st, rs, rsz,
                               next + 1, g->off.p, g->adj.p, T.p, tmark.p, tlist.p, alist.p, ag.p, amask.p, aend.p,
                               chunks.p, hmin.p, dcw.p, S, ctr.p);
            const uint32_t R = std::min(kWRoundsAhead, *std::max_element(hist, hist + kRoundHistory));
            launched[next % kWRing] = R;
            rounds(next, 0, R);
            filter(next, touched, 1u, (R + 1) & 1u);
            commit(next, touched);
            PADO_HIP(hipEventRecord(ev[next % kWRing], st));
        }
        PADO_HIP(hipEventSynchronize(ev[b % kWRing]));
        PADO_HIP(hipGetLastError());
        if (ring[b % kWRing].held) {
            idx->holds += 1;
            hipLaunchKernelGGL(k_w_unhold, dim3(1), dim3(1), 0, st, ctr.p);
            uint32_t done = launched[b % kWRing], more = 1;
            for (;;) {
                PADO_HIP(hipMemcpyAsync(h, ctr.p, sizeof(WCounters), hipMemcpyDeviceToHost, st));
                PADO_HIP(hipStreamSynchronize(st));
                if (!h->n_act[(done + 1) & 1u]) break;  // no frontier for the next round
                rounds(b, done, more);
                done += more;
                more = std::min(2 * more, 64u);
            }
            const u64 labels_before = h->labels;
            filter(b, h->n_touched, 0u, 0u);
            // The touched vertices are known once the rounds end: when even the
            // reservation bound fits the pool, the commit needs no host check.
            bool grow = h->pool_top + h->need_bound > pool_size;
            if (grow) {
                PADO_HIP(hipMemcpyAsync(h, ctr.p, sizeof(WCounters), hipMemcpyDeviceToHost, st));
                PADO_HIP(hipStreamSynchronize(st));
                grow = h->pool_top + h->need > pool_size;
            }
            if (grow) {
                idx->grows += 1;
                idx->pool_words = std::max<uint64_t>(idx->pool_words, h->pool_top);
                // Compact every list into a larger pool.  After compaction a list of
                // length L has capacity L + L/4 + 4, so the commit can reserve at
                // most 2.5 * live + new + 8 * touched words.
                const u64 added = h->labels - labels_before;
                std::vector<uint32_t> hl(n);
                PADO_HIP(copy_sync(hl.data(), len.p, 4ull * n, hipMemcpyDeviceToHost, st));
                std::vector<uint64_t> no(n + 1, 0);
                std::vector<uint32_t> nc(n);
                for (uint32_t v = 0; v < n; ++v) {
                    nc[v] = hl[v] + (hl[v] >> 2) + 4;
                    no[v + 1] = no[v] + nc[v];
                }
                const u64 nsize = std::max<u64>(pool_size * 2, 4 * no[n] + 2 * added + 8ull * h->n_touched + 1024);
                DevBuf<u64> np;
                DevBuf<uint64_t> dno;
                PADO_TRY(np.alloc(nsize, wp));
                PADO_TRY(dno.alloc((uint64_t)n + 1, wp));
                PADO_HIP(copy_sync(dno.p, no.data(), 8ull * (n + 1), hipMemcpyHostToDevice, st));
                hipLaunchKernelGGL(k_w_move, dim3(grid_for((uint64_t)n * 64, 256, 8192)), dim3(256), 0, st, n, pool.p,
                                   base.p, len.p, dno.p, np.p);
                PADO_HIP(hipStreamSynchronize(st));
                std::vector<u64> nb64(no.begin(), no.end() - 1);
                PADO_HIP(copy_sync(base.p, nb64.data(), 8ull * n, hipMemcpyHostToDevice, st));
                PADO_HIP(copy_sync(cap.p, nc.data(), 4ull * n, hipMemcpyHostToDevice, st));
                pool.swap(np);
                pool_size = nsize;
                S.pool = pool.p;
                S.pool_size = pool_size;
                const u64 top = no[n];
                PADO_HIP(copy_sync(&ctr.p->pool_top, &top, 8, hipMemcpyHostToDevice, st));
            }
            commit(b, h->n_touched);
            PADO_HIP(hipStreamSynchronize(st));
            next = b + 1;  // the ones behind it did nothing
        }
        const WClosed done{ring[b % kWRing].rounds, 0u, ring[b % kWRing].n_touched};
        hist[b % kRoundHistory] = (uint32_t)(done.rounds - rounds_seen);
        rounds_seen = done.rounds;
        touched = done.n_touched;
    }
    hipLaunchKernelGGL(k_w_fold_stats, dim3(1), dim3(1024), 0, st, ctr.p);
    PADO_HIP(hipMemcpyAsync(h, ctr.p, sizeof(WCounters), hipMemcpyDeviceToHost, st));
    PADO_HIP(hipStreamSynchronize(st));
    if (h->overflow) {
        set_error("weighted label pool exhausted");
        return PADO_GPU_ERR_NOMEM;
    }
    idx->pool_words = std::max<uint64_t>(idx->pool_words, h->pool_top);
    idx->iterations = h->rounds;
    idx->counters.labels = h->labels;
    idx->counters.pushes = h->relax;
    idx->counters.cands = h->improved;
    idx->counters.dq_pruned = h->pruned;
    idx->counters.bp_pruned = h->filtered;

    // Canonical CSR.  Every list is already sorted by hub: batches commit in
    // root order and k_w_commit writes a batch's roots in ascending order, as
    // the reference's update_index appends them (WPARA:961-990).
    PADO_TRY(idx->loff.alloc((uint64_t)n + 1));
    PADO_TRY(scan_u32_to_u64(len.p, idx->loff.p, n, st, wp));
    uint64_t total = 0;
    PADO_HIP(copy_sync(&total, idx->loff.p + n, 8, hipMemcpyDeviceToHost, st));
    idx->num_labels = total;
    DevBuf<u64> packed;
    PADO_TRY(packed.alloc(total, wp));
    PADO_TRY(idx->whub.alloc(total));
    PADO_TRY(idx->wdist.alloc(total));
    hipLaunchKernelGGL(k_w_move, dim3(grid_for((uint64_t)n * 64, 256, 8192)), dim3(256), 0, st, n, pool.p, base.p,
                       len.p, idx->loff.p, packed.p);
    hipLaunchKernelGGL(k_w_split, dim3(grid_for(total, 256, 8192)), dim3(256), 0, st, total, packed.p, idx->whub.p,
                       idx->wdist.p);
    PADO_HIP(hipStreamSynchronize(st));
    idx->weighted = 1;
    return PADO_GPU_OK;
}

}  // namespace pado
