// query.hip -- exact distance queries over a PADO index on gfx950.
//
// Reference: query_distance, includes/pado_unw_unv_para.201912311607.
// parallel_bp_labeling.h:2283-2416:
//   d = min over the 50 bit-parallel slots of  da + db - {2 | 1 | 0}
//       (2 if S^-1 sets intersect, 1 if S^-1 meets S^0, else 0),
//   d = min(d, min over common hubs h of  La(h) + Lb(h)),
//   d >= 253 -> 255;  ids out of range -> (a == b ? 0 : 255).
// The reference gates each slot with `int td; inti d; if (td - 2 <= d)`,
// an unsigned comparison that skips slots with td < 2 and so over-estimates
// distances from a bit-parallel root to itself and to its neighbours.  The
// default here is the exact (signed) comparison; PADO_GPU_QUERY_REF_COMPAT
// reproduces the reference's answers bit for bit.  Either way the slot order
// does not matter: the result is a minimum over slots.
//
// Mapping: a wave takes up to 64 consecutive pairs.  Lane j reads pair j's ids
// and the tails of their records (label list, component): pairs in different
// components are answered from those alone, the others become jobs in LDS and
// are answered four at a time, sixteen lanes (one DPP row) each, so that the
// first kind leaves no lanes idle.  Pairs with long lists are left to the end
// and take the whole wave, one at a time; so do all pairs of a short call (how
// short goes by the index's mean list length: alone_pairs).
//   Bit-parallel slots: a lane takes four slots as bytes of one word of the
// record.  With m the smallest slot sum, only slots at m or m + 1 can lower
// it, and only where the deciding sets can meet: the record has two bits per
// slot for nonempty sets and S^-1 folded to a byte, so most set pairs are
// never read (46 slots a pair within one of m, 1.8 left, R-MAT 20).
//   Labels: the longer list goes through the group's LDS tile (256 labels,
// padded with all-ones to a power of two), and each lane searches four labels
// of the shorter list in it at once, branch-free.  The reads that need only
// the record's tail go out together: slot words, the longer list's first 128
// labels, the shorter list's first 64; the set pairs are requested next and
// the search runs while they are in flight.  Lists start on 128-byte lines
// and are padded to them with all-ones, so nothing is masked.
// Rank-space queries (many-graph jobs, checks) read the build's own arrays
// through the same code (REC = false).
//
// What bounds it: on a large index the lines read at random (80 M of 128 B for
// 10 M uniform pairs on R-MAT 20: 5.2 TB/s, a copy's rate), on a small one
// instruction issue.  Against one wave per pair with the set pairs of every
// slot within one of m read, in us:
//                                      first   four pairs   records   long alone
//   10 M uniform pairs, R-MAT 20 (HBM) 4,980       4,465     2,325        1,970
//   1 M pairs, half Zipf, R-MAT 14       264         122        87           87
//   2 M pairs, weighted R-MAT 18         742         555       344          341
//   6 M host pairs, R-MAT 18           3,600       2,760     2,190        2,180
// (62% of uniform R-MAT 20 pairs have an isolated end.)
#include "internal.hpp"

namespace pado {
namespace {

constexpr uint32_t kQWaves = 4;               // waves per query block
constexpr uint32_t kQLanes = 16;              // lanes per pair: one DPP row
constexpr uint32_t kQPre = 2;                 // loads of the longer list issued with the first reads
constexpr uint32_t kQBuf = 64 / kQLanes * (16 * kQLanes + 8);  // LDS words per wave
// Waves per SIMD the query kernels are compiled for: five is what their
// registers take without spilling (R-MAT 20 batch: 2,325 us at four or five,
// 2,657 at six).
constexpr int kQOcc = 5;
// Searches a group would do one after the other, from which on the whole wave
// takes the pair instead: it needs one or two, and the wave's other groups
// would have waited for the longest (10 M pairs on R-MAT 20: 1,970 us at 3,
// 2,060 at 2, 2,035 at 4, 2,610 without; weighted R-MAT 18: 364 us at 4, 378
// at 3, 341 without: see kWMixedPairs and kLongMean).
constexpr uint32_t kLongSteps = 3, kWLongSteps = 4;
constexpr uint32_t kNoSlot = 0x7FFFu;         // sum of a slot that does not count

// L lanes work on a pair: a group of a wave, or all of it.
template <uint32_t L>
struct Lanes {
    static constexpr uint32_t kGroups = 64 / L;  // pairs a wave answers at once
    static constexpr uint32_t kTile = 16 * L;    // labels of the longer list held in LDS
    static constexpr uint32_t kStep = 4 * L;     // labels a group moves per load: four per lane
    // Groups' tiles start at different LDS banks: the first search steps of
    // all groups read the same tile position.
    static constexpr uint32_t kStride = kTile + 8;
    static_assert(kGroups * kTile + (kGroups - 1) * 8 <= kQBuf);
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_at4 __attribute__((aligned(4)));  // four words at any word address

template <int N>
__device__ inline uint32_t row_ror(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x120 + N, 0xF, 0xF, false);
}

// The least value of a group's lanes, in all of them.
template <uint32_t L>
__device__ inline uint32_t group_min(uint32_t x)
{
    x = min(x, row_ror<8>(x));
    x = min(x, row_ror<4>(x));
    x = min(x, row_ror<2>(x));
    x = min(x, row_ror<1>(x));
    if constexpr (L == 64) {
        const uint32_t a = __builtin_amdgcn_readlane(x, 0), b = __builtin_amdgcn_readlane(x, 16);
        const uint32_t c = __builtin_amdgcn_readlane(x, 32), d = __builtin_amdgcn_readlane(x, 48);
        x = min(min(a, b), min(c, d));
    }
    return x;
}

// The largest of the groups' values (the same in a group's lanes), as a
// scalar.
template <uint32_t L>
__device__ inline uint32_t groups_max(uint32_t x)
{
    if constexpr (L == 64) return uniform32(x);
    const uint32_t a = __builtin_amdgcn_readlane(x, 0), b = __builtin_amdgcn_readlane(x, kQLanes);
    const uint32_t c = __builtin_amdgcn_readlane(x, 2 * kQLanes), d = __builtin_amdgcn_readlane(x, 3 * kQLanes);
    return max(max(a, b), max(c, d));
}

// Four list entries from position j (any words where j is past the list; see
// mask4).  A read that starts inside the list may run up to three words past
// its end: device buffers have that much slack (DevBuf).
__device__ inline u32x4 load4(const uint32_t *p, uint32_t j, uint32_t len)
{
    u32x4 v = {~0u, ~0u, ~0u, ~0u};
    if (j < len) v = *reinterpret_cast<const u32x4_at4 *>(p + j);
    return v;
}

// The entries of load4 past the list as all-ones, which no label is.  Apart from
// the load, so that a pair's loads are all in flight before the first is
// waited for.
__device__ inline u32x4 mask4(u32x4 v, uint32_t j, uint32_t len)
{
    v.x = j < len ? v.x : ~0u;
    v.y = j + 1 < len ? v.y : ~0u;
    v.z = j + 2 < len ? v.z : ~0u;
    v.w = j + 3 < len ? v.w : ~0u;
    return v;
}

// Lower bounds of four keys in a tile of `size` ascending words (a power of
// two up to TILE): pos[q] = the byte offset of the first word >= key[q], or
// of the last word.  Three vector instructions and an LDS read a step.
template <uint32_t H>
__device__ inline void search_step(const char *tile, uint32_t size, const u32x4 &key, uint32_t (&pos)[4])
{
    if (size > H) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t x = *reinterpret_cast<const uint32_t *>(tile + pos[q] + (4 * H - 4));
            pos[q] = x < key[q] ? pos[q] + 4 * H : pos[q];
        }
    }
    if constexpr (H > 1) search_step<H / 2>(tile, size, key, pos);
}

template <uint32_t TILE>
__device__ inline void search4(const uint32_t *tile, uint32_t size, const u32x4 &key, uint32_t (&pos)[4])
{
#pragma unroll
    for (int q = 0; q < 4; ++q) pos[q] = 0;
    search_step<TILE / 2>(reinterpret_cast<const char *>(tile), size, key, pos);
}

__device__ inline uint32_t tile_at(const uint32_t *tile, uint32_t pos)
{
    return *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(tile) + pos);
}

// A group's four list entries to its tile.
__device__ inline void tile_put(uint32_t *tile, uint32_t j, const u32x4 &v) { *reinterpret_cast<u32x4 *>(tile + j) = v; }

// The power of two at or above x (1 for 0).
__device__ inline uint32_t tile_size(uint32_t x) { return x <= 1u ? 1u : 1u << (32 - __builtin_clz(x - 1u)); }

}  // namespace

// What the query kernels read of an index: the ordered copy's records, or the
// rank-space arrays (rec null).
struct QIndex {
    uint32_t n;
    const uint32_t *rec;
    const uint8_t *bpd;
    const ulonglong2 *bps;
    const uint64_t *loff;
    const uint32_t *lab;    // packed labels, or a weighted index's hubs
    const uint32_t *wdist;  // a weighted index's distances
};

namespace {

// A lane's pair, while it still has to be answered from sets and labels: ids
// and the two label lists, the shorter first.
struct alignas(16) QJob {
    uint32_t a, b;
    uint32_t ls, lt;  // ls: the lane in the top byte (lists have < 2^24 labels)
    uint64_t os, ot;
};

// One wave's LDS.
struct QBuf {
    alignas(16) uint32_t tile[kQBuf];
    QJob job[64];
    uint32_t ans[64];
};

// How a wave's pairs are shared out: all to groups, the ones with long lists
// to the whole wave, or all of them.
enum { kGrouped = 0, kMixed = 1, kAlone = 2 };

// Whether a whole wave takes a pair by itself: where a group would need
// kLongSteps searches or more.
template <bool W>
__device__ inline bool long_lists(uint32_t ls, uint32_t lt)
{
    constexpr uint32_t s = Lanes<kQLanes>::kStep, t = Lanes<kQLanes>::kTile;
    return ((ls + s - 1) / s) * ((lt + t - 1) / t) >= (W ? kWLongSteps : kLongSteps);
}

// Sorts out the wave's pairs (lane j: pair j if `has`): the ones left to
// answer go to buf.job, njobs of them, the first ngroup for groups, the others
// for the whole wave; sets ans to the lane's answer if
// it needs none of that: an id past the index (a == b ? 0 : far), two
// components (far).
template <bool REC, uint32_t RECW, int M>
__device__ inline void make_jobs(const QIndex &X, bool has, uint32_t a, uint32_t b, uint32_t far, QBuf &buf,
                                 uint32_t &ans, bool &job, uint32_t &ngroup, uint32_t &njobs)
{
    const uint32_t lane = threadIdx.x & 63;
    ans = a == b ? 0u : far;
    job = has && a < X.n && b < X.n;
    uint64_t oa = 0, ob = 0;
    uint32_t la = 0, lb = 0;
    if (job) {
        if constexpr (REC) {
            const uint4 ta = *reinterpret_cast<const uint4 *>(X.rec + (uint64_t)a * RECW + (RECW - 4));
            const uint4 tb = *reinterpret_cast<const uint4 *>(X.rec + (uint64_t)b * RECW + (RECW - 4));
            const uint64_t pa = ((uint64_t)ta.w << 32) | ta.z, pb = ((uint64_t)tb.w << 32) | tb.z;
            oa = pa >> 24;
            ob = pb >> 24;
            la = ta.z & 0xFFFFFFu;
            lb = tb.z & 0xFFFFFFu;
            job = ta.y == tb.y;
            if (!job) ans = far;
        } else {
            oa = X.loff[a];
            ob = X.loff[b];
            la = (uint32_t)(X.loff[a + 1] - oa);
            lb = (uint32_t)(X.loff[b + 1] - ob);
        }
    }
    const bool sw = la > lb;
    QJob j;
    j.a = a;
    j.b = b;
    j.os = sw ? ob : oa;
    j.ot = sw ? oa : ob;
    j.ls = (sw ? lb : la) | (lane << 24);
    j.lt = sw ? la : lb;
    const bool alone = M == kAlone || M == kMixed && long_lists<RECW == kWRecWords>(sw ? lb : la, j.lt);
    const unsigned long long mg = __ballot(job && !alone), ma = __ballot(job && alone);
    ngroup = (uint32_t)__popcll(mg);
    njobs = ngroup + (uint32_t)__popcll(ma);
    if (job) buf.job[(alone ? ngroup : 0u) + (uint32_t)__popcll((alone ? ma : mg) & ((1ull << lane) - 1ull))] = j;
    wave_lds_sync();
}

// Answers jobs r0 to njobs, 64 / L at a time, each job's answer to
// buf.ans[its lane].
// Hop<false>: the reference's answers (255 for unreachable or >= 253);
// Hop<true>: exact hops, 0xFFFF for unreachable, using only bit-parallel slots
// reached on both sides.
template <bool W, bool REC, uint32_t L>
__device__ inline void answer_jobs(const QIndex &X, uint32_t r0, uint32_t njobs, bool ref_compat, QBuf &buf)
{
    constexpr uint32_t B = Hop<W>::kBits, MASK = Hop<W>::kInf;
    constexpr uint32_t UNREACHED = W ? 0xFFFFu : 255u;
    using G = Lanes<L>;
    // (the slots take one row of lanes: the rows of a wave that works on one
    // pair all do the same)
    const uint32_t sl = threadIdx.x & (kQLanes - 1);
    const uint32_t lane = threadIdx.x & 63, l = lane & (L - 1), g = lane / L;
    uint32_t *tile = buf.tile + g * G::kStride;
    for (; r0 < njobs; r0 += G::kGroups) {
        // (a group without a job repeats the first one's)
        const bool has = r0 + g < njobs;
        const QJob job = buf.job[has ? r0 + g : r0];
        const uint32_t ls = job.ls & 0xFFFFFFu, lt = job.lt;
        const uint32_t *S = X.lab + job.os, *T = X.lab + job.ot;
        uint32_t wa, wb, fa = 0, fb = 0;
        if constexpr (REC) {
            const uint32_t *pa = X.rec + (uint64_t)job.a * kQRecWords + sl, *pb = X.rec + (uint64_t)job.b * kQRecWords + sl;
            wa = pa[0];
            wb = pb[0];
            fa = pa[kQRecFold];
            fb = pb[kQRecFold];
        } else {
            wa = reinterpret_cast<const uint32_t *>(X.bpd + (uint64_t)job.a * kBpdStride)[sl];
            wb = reinterpret_cast<const uint32_t *>(X.bpd + (uint64_t)job.b * kBpdStride)[sl];
        }
        u32x4 tv[kQPre];
#pragma unroll
        for (uint32_t u = 0; u < kQPre; ++u) tv[u] = load4(T, u * G::kStep + 4 * l, lt);
        const u32x4 s0 = load4(S, 4 * l, ls);
        const uint32_t ms = groups_max<L>(ls), mt = groups_max<L>(lt);
        // This lane's four slots (the last lanes have none).
        uint32_t td[4];
        {
            const uint32_t lo = (wa & 0x00FF00FFu) + (wb & 0x00FF00FFu);
            const uint32_t hi = ((wa >> 8) & 0x00FF00FFu) + ((wb >> 8) & 0x00FF00FFu);
            td[0] = lo & 0xFFFFu;
            td[1] = hi & 0xFFFFu;
            td[2] = lo >> 16;
            td[3] = hi >> 16;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                bool ok = 4 * sl + j < kBP;
                if (W)  // 255: the slot's BFS did not reach this vertex
                    ok = ok && ((wa >> (8 * j)) & 255u) != kInf8 && ((wb >> (8 * j)) & 255u) != kInf8;
                else
                    ok = ok && !(ref_compat && td[j] < 2u);
                if (!ok) td[j] = kNoSlot;
            }
        }
        // Which of this lane's slots can have S^-1 sets that meet (bits of
        // `both`) and which S^-1 on one side and S^0 on the other (`cross`).
        uint32_t both, cross;
        {
            const uint32_t sh = 8 * ((kBpNzByte + sl) & 3u), from = (lane & ~(kQLanes - 1)) + ((kBpNzByte + sl) >> 2);
            const uint32_t na = __shfl(wa, from) >> sh, nb = __shfl(wb, from) >> sh;
            if constexpr (REC) {
                // the bytes of f that are not zero, as four bits
                const uint32_t f = fa & fb;
                const uint32_t h = (((f & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | f) & 0x80808080u;
                both = (h * 0x00204081u) >> 28;
            } else {
                both = na & nb & 15u;
            }
            cross = ((na & (nb >> 4)) | ((na >> 4) & nb)) & 15u;
        }
        const ulonglong2 *ra = X.bps + (uint64_t)job.a * kBP + 4 * sl, *rb = X.bps + (uint64_t)job.b * kBP + 4 * sl;
        if (min(min(td[0], td[1]), min(td[2], td[3])) < 2u) {
            // A sum that its sets would take below zero does not count (no
            // such slot in a built index: a root's own sets are empty).
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                if (td[j] >= 2u || !(((both | cross) >> j) & 1u)) continue;
                const ulonglong2 xa = ra[j], xb = rb[j];
                const uint64_t neg = (xa.x & xb.x) | (td[j] == 0u ? (xa.x & xb.y) | (xa.y & xb.x) : 0ull);
                td[j] = neg ? kNoSlot : td[j];
            }
        }
        const uint32_t m = group_min<L>(min(min(td[0], td[1]), min(td[2], td[3])));
        // The slots at m (cm) and m + 1 (cn) that their sets can lower: S^-1
        // against S^-1 by two, S^-1 against S^0 by one (which does not help
        // at m + 1).
        uint32_t cm, cn;
        {
            uint32_t em = 0, en = 0;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                em |= td[j] == m ? 1u << j : 0u;
                en |= td[j] == m + 1u ? 1u << j : 0u;
            }
            if (m == kNoSlot || sl > (kBP - 1) / 4) em = en = 0u;
            cm = em & (both | cross);
            cn = en & both;
        }
        // The lane's first set pair is requested before the search.
        uint32_t j0 = 0;
        ulonglong2 sa = {0, 0}, sb = {0, 0};
        const bool first = (cm | cn) != 0u, first_m = cm != 0u;
        if (first) {
            j0 = (uint32_t)__builtin_ctz(first_m ? cm : cn);
            sa = ra[j0];
            sb = rb[j0];
            if (first_m)
                cm &= cm - 1u;
            else
                cn &= cn - 1u;
        }
        uint32_t d = m < UNREACHED && m != kNoSlot ? m : UNREACHED;
        for (uint32_t t0 = 0; ms && t0 < mt; t0 += G::kTile) {
            const uint32_t size = tile_size(min(mt - t0, G::kTile));
            for (uint32_t u = 0; u * G::kStep < size; ++u) {
                const uint32_t j = t0 + u * G::kStep + 4 * l;
                const u32x4 v = t0 == 0 && u < kQPre ? (u ? tv[1] : tv[0]) : load4(T, j, lt);
                tile_put(tile, u * G::kStep + 4 * l, REC ? v : mask4(v, j, lt));
            }
            wave_lds_sync();
            for (uint32_t i = 0; i < ms; i += G::kStep) {
                const u32x4 v = i == 0 ? s0 : load4(S, i + 4 * l, ls);
                const u32x4 s = REC ? v : mask4(v, i + 4 * l, ls);
                // A packed label with the same hub is >= the hub with
                // distance 0, so whole words compare as hubs do.
                const u32x4 key = s & ~MASK;
                uint32_t pos[4];
                search4<G::kTile>(tile, size, key, pos);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // x - key is the other distance if the hubs are equal,
                    // else at least MASK + 1.  An entry past its list
                    // (all-ones) has the last hub there can be, but distance
                    // MASK, which no label of that hub has.  A u8 answer
                    // starts at MASK, so neither lowers it.
                    const uint32_t u = tile_at(tile, pos[q]) - key[q], e = s[q] & MASK;
                    const uint32_t sum = __builtin_elementwise_add_sat(u, e);
                    d = min(d, W && max(u, e) >= MASK ? UNREACHED : sum);
                }
            }
            // The next copy must not overtake these reads.
            wave_lds_sync();
        }
        d = group_min<L>(d);
        if (first) {
            if (sa.x & sb.x)
                d = min(d, first_m ? m - 2u : m - 1u);
            else if (first_m && ((sa.x & sb.y) | (sa.y & sb.x)))
                d = min(d, m - 1u);
        }
        // The others, where they can still lower the answer.
        if (d + 1u <= m) cn = 0u, cm &= both;
        if (d + 2u <= m) cm = 0u;
        while (cm | cn) {
            const bool at_m = cm != 0u;
            const uint32_t j = (uint32_t)__builtin_ctz(at_m ? cm : cn);
            const ulonglong2 xa = ra[j], xb = rb[j];
            if (at_m)
                cm &= cm - 1u;
            else
                cn &= cn - 1u;
            if (xa.x & xb.x)
                d = min(d, at_m ? m - 2u : m - 1u);
            else if (at_m && ((xa.x & xb.y) | (xa.y & xb.x)))
                d = min(d, m - 1u);
        }
        d = group_min<L>(d);
        if (!W && d >= 253u) d = 255u;
        if (has && l == 0) buf.ans[job.ls >> 24] = d;
    }
    wave_lds_sync();
}

// Weighted query_distance (WPARA:2125-2243): min over common hubs of
// La(h) + Lb(h).  Exact u32 answers, 0xFFFFFFFF when no hub is shared; with
// ref_compat the reference's int16 domain (>= 32765 -> 32767, ids out of
// range -> a == b ? 0 : 32767).  As answer_jobs, on the hub lists;
// distances of the shorter list come in with its hubs, those of the longer
// list are read where a hub matches.
template <bool REC, uint32_t L>
__device__ inline void answer_wjobs(const QIndex &X, uint32_t r0, uint32_t njobs, bool ref_compat, QBuf &buf)
{
    using G = Lanes<L>;
    const uint32_t lane = threadIdx.x & 63, l = lane & (L - 1), g = lane / L;
    uint32_t *tile = buf.tile + g * G::kStride;
    for (; r0 < njobs; r0 += G::kGroups) {
        const bool has = r0 + g < njobs;
        const QJob job = buf.job[has ? r0 + g : r0];
        const uint32_t ls = job.ls & 0xFFFFFFu, lt = job.lt;
        const uint32_t *S = X.lab + job.os, *T = X.lab + job.ot;
        const uint32_t *DS = X.wdist + job.os, *DT = X.wdist + job.ot;
        u32x4 tv[kQPre];
#pragma unroll
        for (uint32_t u = 0; u < kQPre; ++u) tv[u] = load4(T, u * G::kStep + 4 * l, lt);
        const u32x4 s0 = load4(S, 4 * l, ls), d0 = load4(DS, 4 * l, ls);
        const uint32_t ms = groups_max<L>(ls), mt = groups_max<L>(lt);
        uint32_t d = 0xFFFFFFFFu;
        for (uint32_t t0 = 0; ms && t0 < mt; t0 += G::kTile) {
            const uint32_t size = tile_size(min(mt - t0, G::kTile));
            for (uint32_t u = 0; u * G::kStep < size; ++u) {
                const uint32_t j = t0 + u * G::kStep + 4 * l;
                const u32x4 v = t0 == 0 && u < kQPre ? (u ? tv[1] : tv[0]) : load4(T, j, lt);
                tile_put(tile, u * G::kStep + 4 * l, REC ? v : mask4(v, j, lt));
            }
            wave_lds_sync();
            for (uint32_t i = 0; i < ms; i += G::kStep) {
                const u32x4 v = i == 0 ? s0 : load4(S, i + 4 * l, ls);
                const u32x4 s = REC ? v : mask4(v, i + 4 * l, ls);
                const u32x4 e = i == 0 ? d0 : load4(DS, i + 4 * l, ls);
                uint32_t pos[4], x[4];
                search4<G::kTile>(tile, size, s, pos);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    x[q] = 0xFFFFFFFFu;
                    if (tile_at(tile, pos[q]) == s[q] && s[q] != ~0u) x[q] = DT[t0 + pos[q] / 4];
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)  // (no hub, or a sum past 2^32: all-ones, which lowers nothing)
                    d = min(d, __builtin_elementwise_add_sat(x[q], e[q]));
            }
            wave_lds_sync();
        }
        d = group_min<L>(d);
        if (ref_compat && d >= 32765u) d = 32767u;
        if (has && l == 0) buf.ans[job.ls >> 24] = d;
    }
    wave_lds_sync();
}

// Kinds of index: u8 hops, the wide hop domain, weighted.
enum { kHops = 0, kWideHops = 1, kWeights = 2 };

// Answers the wave's pairs, lane j holding pair j if `has`; returns the lane's
// answer.
template <int K, bool REC, int M>
__device__ inline uint32_t answer_pairs(const QIndex &X, bool has, uint32_t a, uint32_t b, bool ref_compat, QBuf &buf)
{
    const uint32_t far = K == kHops ? 255u : K == kWideHops ? 0xFFFFu : ref_compat ? 32767u : 0xFFFFFFFFu;
    uint32_t ans;
    bool job;
    uint32_t ngroup, njobs;
    make_jobs<REC, K == kWeights ? kWRecWords : kQRecWords, M>(X, has, a, b, far, buf, ans, job, ngroup, njobs);
    if constexpr (K == kWeights) {
        if constexpr (M != kAlone) answer_wjobs<REC, kQLanes>(X, 0, ngroup, ref_compat, buf);
        if constexpr (M != kGrouped) answer_wjobs<REC, 64>(X, ngroup, njobs, ref_compat, buf);
    } else {
        if constexpr (M != kAlone) answer_jobs<K == kWideHops, REC, kQLanes>(X, 0, ngroup, ref_compat, buf);
        if constexpr (M != kGrouped) answer_jobs<K == kWideHops, REC, 64>(X, ngroup, njobs, ref_compat, buf);
    }
    return job ? buf.ans[threadIdx.x & 63] : ans;
}

}  // namespace

// Batch queries: a wave takes `chunk` consecutive pairs at a time (see
// query_chunk).  OT: the answer type (u16 for a wide index or widened
// answers).
template <int K, bool REC, int M, class OT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kQOcc))) void k_query(QIndex X, const uint32_t *qa,
                                               const uint32_t *qb, uint64_t k, uint32_t chunk, OT *out,
                                               int ref_compat)
{
    __shared__ QBuf s_q[kQWaves];
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t nw = ((uint64_t)gridDim.x * blockDim.x) >> 6;
    const uint64_t w = uniform64(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    for (uint64_t c0 = w * chunk; c0 < k; c0 += nw * chunk) {
        const bool has = lane < chunk && c0 + lane < k;
        const uint32_t a = has ? qa[c0 + lane] : 0u, b = has ? qb[c0 + lane] : 0u;
        const uint32_t d = answer_pairs<K, REC, M>(X, has, a, b, ref_compat != 0, s_q[threadIdx.x >> 6]);
        if (has) out[c0 + lane] = (OT)d;
        // The next chunk's jobs and answers must not overtake these reads.
        wave_lds_sync();
    }
}

// Persistent label-merge kernels for the serving loop: a grid sized to the
// chip's resident waves; each wave takes kGrab pairs at a time from a
// per-launch work counter until the launch's k pairs are exhausted, so waves
// that draw long label lists do not hold back the launch.  Every wave leaves
// once the counter passes k.
constexpr uint32_t kGrab = 16;

template <int K, int M, class OT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kQOcc))) void k_query_ws(QIndex X, const uint32_t *qa,
                                                  const uint32_t *qb, uint64_t k, OT *out, int ref_compat,
                                                  unsigned long long *work)
{
    __shared__ QBuf s_q[kQWaves];
    const uint32_t lane = threadIdx.x & 63;
    for (;;) {
        unsigned long long c0 = 0;
        if (lane == 0) c0 = atomicAdd(work, (unsigned long long)kGrab);
        c0 = uniform64(c0);
        if (c0 >= k) break;
        const bool has = lane < kGrab && c0 + lane < k;
        const uint32_t a = has ? qa[c0 + lane] : 0u, b = has ? qb[c0 + lane] : 0u;
        const uint32_t d = answer_pairs<K, true, M>(X, has, a, b, ref_compat != 0, s_q[threadIdx.x >> 6]);
        if (has) out[c0 + lane] = (OT)d;
        wave_lds_sync();
    }
}

__global__ void k_zero_work(unsigned long long *work) { *work = 0ull; }

// Resident workgroups per CU of the persistent kernel: the label merge waits
// on dependent loads, so the grid fills every slot the kernel's registers and
// LDS leave (a fixed 4 per CU left serving at 70% of the grid-stride kernel).
uint32_t query_ws_blocks_per_cu(bool weighted)
{
    int nb = 0;
    const hipError_t e = weighted ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_query_ws<kWeights, kMixed, uint32_t>, 256, 0)
                                  : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_query_ws<kHops, kMixed, uint8_t>, 256, 0);
    return (e == hipSuccess && nb > 0) ? (uint32_t)nb : 4u;
}

// ---------------------------------------------------------------------------
// Resident serving kernel.  One launch stays on the device while requests
// flow: the host writes a request's pairs into the mapped ring, cuts them
// into descriptors of at most kServeGroup pairs spread over kServeQueues
// queues, and raises each queue's published count in mapped memory.  Wave 0
// of workgroup 0 polls those counts (one host read per queue per round) and
// mirrors them into device memory; every other wave takes tickets from its
// queue's device counter (queues are picked by workgroup, so the eight
// counters and their traffic spread over the XCDs) and waits, sleeping, on
// the mirrored count in L2.  A wave answers its descriptor's pairs with the
// label merge of the batch kernel (answer_pairs): one host read brings in the
// up-to-64 pairs' ids (lane j holds pair j), the lanes sort their own pairs
// into jobs in LDS, and groups of lanes or the whole wave answer these; the
// answers go back as one contiguous store into the mapped answer ring.  The
// wave that completes a request's last descriptor writes the request's
// sequence number into its slot's completion flag.  The poller stops taking in
// new descriptors once asked to (host stop flag), after max_ticks in any case,
// or after idle_ticks without work; when every descriptor taken in is done it
// raises the exit flag, and every wave leaves.  The host relaunches the kernel
// when work arrives after an exit.
namespace {

// Relaxed device-coherent load.  No acquire anywhere in the serving loop: an
// acquire at device scope invalidates the L2, and thousands of polling waves
// doing that would strip the cache from the waves that answer queries.
// Nothing a wave reads after a poll can be stale without it: the descriptors,
// pairs and answers are in uncached host memory, read and written with
// system-scope accesses, and the index does not change while it is served.
__device__ inline unsigned long long ld_agent(unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class T>
__device__ inline T ld_sys(const T *p)
{
    return __hip_atomic_load(const_cast<T *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <class T>
__device__ inline void st_sys(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Waits until this wave's earlier memory operations (stores included) are done.
__device__ inline void wait_memory() { __builtin_amdgcn_s_waitcnt(0); }

// The value of the wave's first active lane, as a wave-uniform (scalar)
// value.  Every control decision of the serving loop goes through it: the
// compiler must see the ticket, the published count, the exit flag and the
// descriptor as uniform, or it structures the loops for lanes that could
// part ways -- and a lane set that re-enters the wait without lane 0 would
// broadcast a stale ticket.
// (uniform64 / uniform32: common.hpp)

__device__ void serve_poll(const ServeKernelArgs &A)
{
    const uint32_t lane = threadIdx.x & 63;
    unsigned long long *S = A.state;
    uint64_t *pub = const_cast<uint64_t *>(A.ctl->pub);
    uint32_t *stop_p = const_cast<uint32_t *>(&A.ctl->stop);
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    uint64_t last = t0;
    bool frozen = false;
    for (;;) {
        const uint64_t now = __builtin_amdgcn_s_memrealtime();
        const uint32_t stop = uniform32(ld_sys(stop_p));
        bool moved = false, busy = false;
        if (lane < kServeQueues) {
            unsigned long long seen = ld_agent(&S[serve_seen(lane)]);
            if (!frozen) {
                const uint64_t p = ld_sys(pub + lane);
                if (p > seen) {
                    __hip_atomic_store(&S[serve_seen(lane)], (unsigned long long)p, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                    seen = p;
                    moved = true;
                }
            }
            busy = ld_agent(&S[serve_done(lane)]) != seen;
        }
        const bool any_busy = __ballot(busy) != 0ull;
        if (__ballot(moved) != 0ull || any_busy) last = now;
        if (stop || now - t0 > A.max_ticks || (!any_busy && now - last > A.idle_ticks)) frozen = true;
        if (frozen && !any_busy) {
            __hip_atomic_store(&S[kServeExit], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        __builtin_amdgcn_s_sleep(16);
    }
}

template <int K>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kQOcc))) void k_serve(QIndex X, ServeKernelArgs A)
{
    __shared__ QBuf s_q[kQWaves];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (blockIdx.x == 0 && wv == 0) {
        serve_poll(A);
        return;
    }
    unsigned long long *S = A.state;
    const uint32_t q = blockIdx.x % kServeQueues;
    for (;;) {
        // Every lane takes part in the loop's atomics with lane 0 alone
        // contributing (no lane-0-only branch for the loop structure to split
        // on); lane 0 is the first active lane, so its result is the ticket.
        const uint64_t c = uniform64(atomicAdd(&S[serve_claim(q)], lane == 0 ? 1ull : 0ull));
        bool leave = false;
        for (;;) {
            if (uniform64(ld_agent(&S[serve_seen(q)])) > c) break;
            if (uniform64(ld_agent(&S[kServeExit])) != 0) {
                leave = true;
                break;
            }
            // About a microsecond between polls: waiting waves stay off the
            // memory system the working ones use.
            __builtin_amdgcn_s_sleep(40);
        }
        if (leave) return;
        // The descriptor and the pairs live in mapped host memory that is
        // not cached on the device.
        ServeDesc *dp = const_cast<ServeDesc *>(A.desc) + (uint64_t)q * A.dcap + c % A.dcap;
        const uint64_t pos = uniform64(ld_sys(&dp->pos));
        const uint32_t len = uniform32(ld_sys(&dp->len));
        const uint32_t slot = uniform32(ld_sys(&dp->slot));
        const uint64_t seq = uniform64(ld_sys(&dp->seq));
        const uint32_t rk = uniform32(ld_sys(&dp->k));
        const uint64_t phys = pos % A.cap;
        uint32_t ia = 0, ib = 0;
        if (lane < len) {
            ia = ld_sys(A.ra + phys + lane);
            ib = ld_sys(A.rb + phys + lane);
        }
        const uint32_t mine = answer_pairs<K, true, kMixed>(X, lane < len, ia, ib, A.ref_compat != 0, s_q[wv]);
        // The next descriptor's writes must not overtake these reads.
        wave_lds_sync();
        if (lane < len) {
            if (K == kHops) st_sys(static_cast<uint8_t *>(A.out) + phys + lane, (uint8_t)mine);
            if (K == kWideHops) st_sys(static_cast<uint16_t *>(A.out) + phys + lane, (uint16_t)mine);
            if (K == kWeights) st_sys(static_cast<uint32_t *>(A.out) + phys + lane, mine);
        }
        // The answers have reached host memory before this wave's count
        // moves (the stores write through to the host; waiting for them is
        // all the ordering they need).
        wait_memory();
        const uint32_t prev = uniform32(__hip_atomic_fetch_add(&A.rdone[slot], lane == 0 ? len : 0u,
                                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (prev + len == rk) {
            // Last descriptor of the request: reset the slot's count (the
            // host reuses the slot only after it sees the flag), then raise
            // the flag.  Every lane stores the same value.
            __hip_atomic_store(&A.rdone[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            wait_memory();
            st_sys(A.flags + slot, seq);
            wait_memory();
        }
        __hip_atomic_fetch_add(&S[serve_done(q)], lane == 0 ? 1ull : 0ull, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Start of a launch: the previous launch exited only once every descriptor
// it took in was done, so tickets restart at the done count.
__global__ void k_serve_reset(unsigned long long *S)
{
    const uint32_t q = threadIdx.x;
    if (q < kServeQueues) S[serve_claim(q)] = S[serve_done(q)];
    if (q == 0) S[kServeExit] = 0ull;
}

}  // namespace

uint32_t serve_resident_blocks_per_cu(const pado_gpu_index *idx)
{
    int nb = 0;
    hipError_t e;
    if (idx->weighted)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_serve<kWeights>, 256, 0);
    else if (idx->wide)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_serve<kWideHops>, 256, 0);
    else
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_serve<kHops>, 256, 0);
    return (e == hipSuccess && nb > 0) ? (uint32_t)nb : 4u;
}

// The ordered copy of an index (or its rank-space arrays).
static QIndex query_index(const pado_gpu_index *idx, bool rank_space)
{
    QIndex X{};
    X.n = idx->n;
    if (rank_space) {
        X.bpd = idx->bpd.p;
        X.bps = (const ulonglong2 *)idx->bps.p;
        X.loff = idx->loff.p;
        X.lab = idx->weighted ? idx->whub.p : idx->lab.p;
        X.wdist = idx->wdist.p;
    } else {
        X.rec = idx->qrec.p;
        X.bps = (const ulonglong2 *)idx->qbps.p;
        X.lab = idx->qlab.p;
        X.wdist = idx->qwdist.p;
    }
    return X;
}

pado_gpu_status launch_serve_resident(const pado_gpu_index *idx, const ServeKernelArgs &a, uint32_t blocks,
                                      hipStream_t st)
{
    const QIndex X = query_index(idx, false);
    hipLaunchKernelGGL(k_serve_reset, dim3(1), dim3(64), 0, st, a.state);
    if (idx->weighted)
        hipLaunchKernelGGL(k_serve<kWeights>, dim3(blocks), dim3(256), 0, st, X, a);
    else if (idx->wide)
        hipLaunchKernelGGL(k_serve<kWideHops>, dim3(blocks), dim3(256), 0, st, X, a);
    else
        hipLaunchKernelGGL(k_serve<kHops>, dim3(blocks), dim3(256), 0, st, X, a);
    PADO_HIP(hipGetLastError());
    return PADO_GPU_OK;
}

// One pair, ids passed by value, the answer written into mapped host memory
// with a system-scope store: a lone query costs one launch and one stream
// synchronisation, no copies.
template <int K, bool REC>
__global__ __launch_bounds__(64) void k_query_pair(QIndex X, uint32_t a, uint32_t b, int ref_compat, uint32_t *out)
{
    __shared__ QBuf buf;
    const uint32_t d = answer_pairs<K, REC, kAlone>(X, threadIdx.x == 0, a, b, ref_compat != 0, buf);
    if (threadIdx.x == 0) __hip_atomic_store(out, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int K>
static void launch_pair(const QIndex &X, uint32_t a, uint32_t b, bool ref, uint32_t *out_dev, hipStream_t st)
{
    if (X.rec)
        hipLaunchKernelGGL((k_query_pair<K, true>), dim3(1), dim3(64), 0, st, X, a, b, ref ? 1 : 0, out_dev);
    else
        hipLaunchKernelGGL((k_query_pair<K, false>), dim3(1), dim3(64), 0, st, X, a, b, ref ? 1 : 0, out_dev);
}

pado_gpu_status launch_query_pair(const pado_gpu_index *idx, bool rank_space, uint32_t a, uint32_t b,
                                  bool ref_compat, uint32_t *out_dev, hipStream_t st)
{
    const QIndex X = query_index(idx, rank_space);
    if (idx->weighted)
        launch_pair<kWeights>(X, a, b, ref_compat, out_dev, st);
    else if (idx->wide)
        launch_pair<kWideHops>(X, a, b, false, out_dev, st);
    else
        launch_pair<kHops>(X, a, b, ref_compat, out_dev, st);
    PADO_HIP(hipGetLastError());
    return PADO_GPU_OK;
}

namespace {

// How a call's pairs are shared out goes by the pairs and by the index's mean
// list length: R-MAT graphs have 2 to 80 labels a vertex (weighted 20 to 220),
// grids 30 to 170, sparse random graphs of 20 K to 200 K vertices 300 to 2,800.
//
// Up to so many pairs a whole wave takes each: the waves are on the chip
// together, and a call takes as long as its longest lists, which the wave goes
// through in fewer steps.  In us, alone against groups or the mix:
//   mean 22-34,   6,000 pairs: 5.5-6.8 and 4.4-5.9 (3,000: equal)
//   mean 80-170,  6,000: 5.8-7.1 and 9.2-10.1;  12,000: 8.1-10.9 and 9.8-14.9;
//                 20,000: 14-18 and 11-18.5
//   mean 300-2,800, 6,000: 10-142 and 15-388;  50,000: 53-918 and 52-4,391;
//                 1,000,000: 0.94-16.8 ms and 0.73-15.3
inline uint64_t alone_pairs(uint32_t mean) { return mean < 64 ? 4096 : mean < 256 ? 12288 : 65536; }

// From this mean on nearly every pair is one for the whole wave, and a
// weighted call takes the mix whatever its size (1 M pairs: 0.96-15.3 ms, in
// groups 1.6-67).  Below it weighted pairs go to groups from kWMixedPairs on:
// the whole wave's part costs registers and scheduling (2 M pairs: 341 us, 362
// mixed) and only a call's last waves gain by it (16,000 pairs: 10.4 us, 9.3
// mixed).
constexpr uint32_t kLongMean = 256;
constexpr uint64_t kWMixedPairs = 32768;

// Consecutive pairs per wave otherwise: as many as leave 8,192 waves work, in
// [4, 64].  A chunk's ids and records are two dependent reads before its first
// pair, so long calls take 64 (1 M pairs: 87 us against 97 with 16 and 161
// with 4); short ones spread over the chip.  Where the pairs come out one
// after the other, 32,768 waves (100,000 pairs: 0.11-1.77 ms with 4, 0.14-2.3
// with 16; 1 M: 0.96-15.3 with 16, 1.06-17.3 with 64).
inline uint32_t query_chunk(uint64_t k, uint32_t mean)
{
    const uint64_t waves = mean < kLongMean ? 8192 : 32768;
    uint32_t c = 64 / kQLanes;
    while (c < 64 && (uint64_t)c * 2 * waves <= k) c *= 2;
    return c;
}

inline uint32_t mean_list(const pado_gpu_index *idx) { return (uint32_t)(idx->num_labels / idx->n); }

template <int K, class OT>
pado_gpu_status launch_batch(const pado_gpu_index *idx, bool rank_space, const uint32_t *qa, const uint32_t *qb,
                             uint64_t k, OT *out, bool ref, hipStream_t st)
{
    if (k == 0) return PADO_GPU_OK;
    const QIndex X = query_index(idx, rank_space);
    const uint32_t mean = mean_list(idx);
    const bool alone = k <= alone_pairs(mean);
    const uint32_t chunk = alone ? 1u : query_chunk(k, mean), grid = grid_for((k + chunk - 1) / chunk * 64, 256, 1u << 20);
    auto kern = X.rec ? (alone ? k_query<K, true, kAlone, OT> : k_query<K, true, kMixed, OT>)
                      : (alone ? k_query<K, false, kAlone, OT> : k_query<K, false, kMixed, OT>);
    if (K == kWeights && k > kWMixedPairs && mean < kLongMean)
        kern = X.rec ? k_query<K, true, kGrouped, OT> : k_query<K, false, kGrouped, OT>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, st, X, qa, qb, k, chunk, out, ref ? 1 : 0);
    PADO_HIP(hipGetLastError());
    return PADO_GPU_OK;
}

}  // namespace

pado_gpu_status launch_wquery(const pado_gpu_index *idx, bool rank_space, const uint32_t *qa, const uint32_t *qb,
                              uint64_t k, uint32_t *out, bool ref_compat, hipStream_t st)
{
    return launch_batch<kWeights>(idx, rank_space, qa, qb, k, out, ref_compat, st);
}

pado_gpu_status launch_query(const pado_gpu_index *idx, bool rank_space, const uint32_t *qa, const uint32_t *qb,
                             uint64_t k, uint8_t *out, bool ref_compat, hipStream_t st)
{
    return launch_batch<kHops>(idx, rank_space, qa, qb, k, out, ref_compat, st);
}

// u16 answers on device pairs: exact hops for a wide index, the reference's
// answers widened for one in the u8 domain.
pado_gpu_status launch_query_wide(const pado_gpu_index *idx, bool rank_space, const uint32_t *qa, const uint32_t *qb,
                                  uint64_t k, uint16_t *out, bool ref_compat, hipStream_t st)
{
    if (idx->wide) return launch_batch<kWideHops>(idx, rank_space, qa, qb, k, out, false, st);
    return launch_batch<kHops>(idx, rank_space, qa, qb, k, out, ref_compat, st);
}

// Query launch on device pairs for either index type, ordered ids: out holds
// u8, u16 (wide) or u32 (weighted) answers.  work == nullptr selects the batch
// kernel; otherwise the persistent kernel with `blocks` workgroups, its
// counter cleared on the same stream first (a wide index always takes the
// batch kernel).
pado_gpu_status launch_query_any(const pado_gpu_index *idx, const uint32_t *qa, const uint32_t *qb, uint64_t k,
                                 void *out, bool ref_compat, hipStream_t st, unsigned long long *work, uint32_t blocks)
{
    if (k == 0) return PADO_GPU_OK;
    if (idx->wide) return launch_query_wide(idx, false, qa, qb, k, (uint16_t *)out, false, st);
    if (!work) {
        if (idx->weighted) return launch_wquery(idx, false, qa, qb, k, (uint32_t *)out, ref_compat, st);
        return launch_query(idx, false, qa, qb, k, (uint8_t *)out, ref_compat, st);
    }
    const uint64_t need = (k + kGrab - 1) / kGrab;  // grabs; one wave per grab at most
    uint32_t grid = blocks;
    if ((uint64_t)grid * 4 > need) grid = (uint32_t)((need + 3) / 4);
    if (grid == 0) grid = 1;
    const QIndex X = query_index(idx, false);
    hipLaunchKernelGGL(k_zero_work, dim3(1), dim3(1), 0, st, work);
    if (idx->weighted)
        hipLaunchKernelGGL((mean_list(idx) < kLongMean ? k_query_ws<kWeights, kGrouped, uint32_t>
                                                       : k_query_ws<kWeights, kMixed, uint32_t>),
                           dim3(grid), dim3(256), 0, st, X, qa, qb, k, (uint32_t *)out, ref_compat ? 1 : 0, work);
    else
        hipLaunchKernelGGL((k_query_ws<kHops, kMixed, uint8_t>), dim3(grid), dim3(256), 0, st, X, qa, qb, k,
                           (uint8_t *)out, ref_compat ? 1 : 0, work);
    PADO_HIP(hipGetLastError());
    return PADO_GPU_OK;
}

}  // namespace pado
