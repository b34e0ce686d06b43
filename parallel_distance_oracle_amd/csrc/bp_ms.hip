// bp_ms.hip -- bit-parallel labeling with all 50 slots in one level-synchronous
// sweep (multi-source BFS), gfx950.
//
// Reference: bit_parallel_labeling, includes/pado_unw_unv_para.201912311607.
// parallel_bp_labeling.h:544-840 (semantics restated in bp.hip's header).  The
// 50 BFSes are independent once the roots and their selected neighbours are
// chosen (a serial host pass, PARA:670-709), so they advance together: a
// vertex carries a 64-bit mask of the slots in which it sits on the current
// level, and one pass over its adjacency serves every such slot.  A vertex is
// expanded once per distinct level it has across the slots (typically 2-4 on
// R-MAT graphs) instead of once per slot.
//
// Per level d two kernels.  A wave takes a 64-edge piece of a vertex's
// adjacency, or four vertices of up to 16 edges; its lanes first take an edge
// each, then, vertex by vertex, a slot each:
//   k_ms_scan(d)  over the level's vertices v: S^0[v][i] |= S^-1[u][i] for
//                 edges (v,u), u != v, both at level d in slot i; slots where
//                 v is at d and u is unvisited put u on level d + 1
//   k_ms_pull(d)  over the new level's vertices u: bp_dist = d + 1, and S^-1,
//                 S^0 of u gather those of its parents (v at d where u is at
//                 d + 1)
// Finally S^0 is masked with ~S^-1 (PARA:829-835, k_bp_finish).  The order
// siblings, then children matches PARA:783-813; set unions are order-free, so
// the records are deterministic.
//
// Masks and vertex lists rotate over three buffers: level L's mask, empty when
// k_ms_scan(L - 1) starts, is cleared by k_ms_pull(L + 1).  Counts are kept per
// level, so the host enqueues levels in growing blocks and reads the counts
// once per block; a level past the last one is two empty launches.
//
// What bounds it: the 800-byte set rows read per (edge, level), 128 B at a
// time; on deep graphs, the chain of dependent reads of a short level.  On R-MAT
// 20 the two kernels of the heaviest level take 3.4 + 1.4 ms, the phase 6.6 ms
// (sets pushed along edges -- one edge per lane, a 64-bit atomic per slot and
// set, two atomics on one counter per new vertex, a host check per level --
// took 9.9 + 9.1 and 24).  A 161 x 161 grid, 255 levels: build 64.6 -> 54.4 ms;
// with one wave per vertex whatever its degree 61.9, since every wave's new
// vertices queue on the level's counters.
#include "internal.hpp"

namespace pado {
namespace {

using u64 = unsigned long long;

constexpr uint32_t kMsPiece = 64;     // edges of a work piece: one per lane
constexpr uint32_t kMsSmall = 16;     // vertices of up to this degree go four to a wave
constexpr uint32_t kMsLevels = 256;   // levels 0..255 can be populated
constexpr uint32_t kMsLine = 32;      // u32 per counter line
constexpr uint32_t kMsAhead = 4;      // set rows in flight per wave

// Vertices of each level, and work pieces of those of degree above kMsSmall, a
// line per counter.
struct MsCounts {
    uint32_t v[kMsLevels + 1][kMsLine], piece[kMsLevels + 1][kMsLine];
};

// One level's view of the sweep (device pointers).
struct MsLevel {
    u64 *cur, *nxt, *old;  // masks of levels d, d + 1, d - 1 (k_ms_pull empties the last)
    const uint32_t *cur_list, *old_list;
    uint32_t *nxt_list;
    const u64 *cur_piece;  // pieces of level d: (edge offset << 32) | vertex
    u64 *nxt_piece;
    MsCounts *cnt;
    uint32_t d;
};

// Lanes with `isnew` put vertex u, of degree deg, on a level's list, and its
// pieces on the level's piece list.  Every lane of the wave calls it.
__device__ inline void ms_emit(bool isnew, uint32_t u, uint32_t deg, uint32_t *list, u64 *pieces, uint32_t *cnt_v,
                               uint32_t *cnt_piece)
{
    if (__ballot(isnew) == 0ull) return;
    const uint32_t at = wave_append(cnt_v, isnew);
    if (isnew) list[at] = u;
    const uint32_t np = isnew && deg > kMsSmall ? (deg + kMsPiece - 1) / kMsPiece : 0u;
    const uint32_t incl = wave_incl_scan(np);
    const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
    if (total == 0) return;
    uint32_t base = 0;
    if ((threadIdx.x & 63) == 0) base = atomicAdd(cnt_piece, total);
    base = uniform32(base) + incl - np;
    for (uint32_t q = 0; q < np; ++q) pieces[base + q] = ((u64)(q * kMsPiece) << 32) | u;
}

// Seeds: roots at level 0 (cur), selected neighbours at level 1 (nxt, vis,
// S^-1 bit).  seeds[j] = (vertex, slot, neighbour index or 255 for the root).
__global__ __launch_bounds__(256) void k_ms_seed(uint32_t nseeds, const uint32_t *seed_v, const uint32_t *seed_slot,
                                                 const uint32_t *seed_j, const uint64_t *off, uint8_t *bpd,
                                                 ulonglong2 *bps, u64 *vis, u64 *nz1, uint32_t *cur_list, u64 *cur_piece,
                                                 MsLevel L)
{
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t s0 = blockIdx.x * blockDim.x + (threadIdx.x & ~63u); s0 < nseeds; s0 += stride) {
        const uint32_t s = s0 + (threadIdx.x & 63);
        bool root = false, first = false;
        uint32_t v = 0, deg = 0;
        if (s < nseeds) {
            v = seed_v[s];
            deg = (uint32_t)(off[v + 1] - off[v]);
            const uint32_t i = seed_slot[s], j = seed_j[s];
            const u64 bit = 1ull << i;
            root = j == 255u;
            atomicOr(&vis[v], bit);
            if (root) {
                bpd[(uint64_t)v * kBpdStride + i] = 0;
                first = atomicOr(&L.cur[v], bit) == 0ull;
            } else {
                bps[(uint64_t)v * kBP + i].x = 1ull << j;
                atomicOr(&nz1[v], bit);
                first = atomicOr(&L.nxt[v], bit) == 0ull;
            }
        }
        ms_emit(first && root, v, deg, cur_list, cur_piece, L.cnt->v[0], L.cnt->piece[0]);
        ms_emit(first && !root, v, deg, L.nxt_list, L.nxt_piece, L.cnt->v[1], L.cnt->piece[1]);
    }
}

// For every lane j of `act`: f(vertex u of lane j, whether this lane's slot is
// in its mask m), kMsAhead of them at a time.
template <class F>
__device__ inline void ms_rows(u64 act, uint32_t u, u64 m, F f)
{
    const uint32_t lane = threadIdx.x & 63;
    while (act) {
        uint32_t w[kMsAhead];
        bool mine[kMsAhead];
#pragma unroll
        for (uint32_t k = 0; k < kMsAhead; ++k) {
            mine[k] = false;
            w[k] = 0;
            if (act) {
                const uint32_t j = (uint32_t)__ffsll(act) - 1;
                act &= act - 1;
                w[k] = __builtin_amdgcn_readlane(u, j);
                mine[k] = (readlane64(m, j) >> lane) & 1ull;
            }
        }
        f(w, mine);
    }
}

template <uint32_t G>
__device__ inline u64 group_lanes(uint32_t g)  // lanes of group g of G
{
    return (G == 64 ? ~0ull : (1ull << (G & 63u)) - 1ull) << (g * G);
}

// k_ms_scan for edges e of vertex v, G lanes per vertex (v: kEmpty if the
// group has none).
template <uint32_t G>
__device__ inline void ms_scan_unit(uint32_t v, uint32_t e, const uint64_t *off, const uint32_t *adj, const u64 *vis,
                                    const u64 *nz1, ulonglong2 *bps, const MsLevel &L)
{
    const uint32_t lane = threadIdx.x & 63;
    uint32_t u = 0, deg = 0, udeg = 0;
    u64 sib = 0ull, child = 0ull;
    if (v != kEmpty) {
        const uint64_t b = off[v];
        deg = (uint32_t)(off[v + 1] - b);
        if (G < 64 && deg > G) deg = 0;  // (its pieces are on the piece list)
        const u64 fv = L.cur[v];
        if (e < deg) {
            u = adj[b + e];
            const u64 fu = L.cur[u], vu = vis[u], n1 = nz1[u];
            child = fv & ~vu;  // (v itself is visited)
            if (u != v) sib = fv & fu & n1;
        }
    }
    bool isnew = false;
    if (child && (child & ~L.nxt[u])) {
        isnew = atomicOr(&L.nxt[u], child) == 0ull;
        if (isnew) udeg = (uint32_t)(off[u + 1] - off[u]);
    }
    ms_emit(isnew, u, udeg, L.nxt_list, L.nxt_piece, L.cnt->v[L.d + 1], L.cnt->piece[L.d + 1]);
    const u64 all = __ballot(sib != 0ull);
    if (!all) return;
    for (uint32_t g = 0; g < 64 / G; ++g) {
        const u64 act = all & group_lanes<G>(g);
        if (!act) continue;
        u64 x = 0ull;
        ms_rows(act, u, sib, [&](const uint32_t (&w)[kMsAhead], const bool (&mine)[kMsAhead]) {
            u64 y[kMsAhead];
#pragma unroll
            for (uint32_t k = 0; k < kMsAhead; ++k) y[k] = mine[k] ? bps[(uint64_t)w[k] * kBP + lane].x : 0ull;
#pragma unroll
            for (uint32_t k = 0; k < kMsAhead; ++k) x |= y[k];
        });
        const uint32_t vg = __builtin_amdgcn_readlane(v, g * G), dg = __builtin_amdgcn_readlane(deg, g * G);
        if (x) {
            ulonglong2 *r = &bps[(uint64_t)vg * kBP + lane];
            if (dg <= G)
                r->y |= x;  // vg's only piece
            else
                atomicOr(&r->y, x);
        }
    }
}

// k_ms_pull for edges e of vertex u, G lanes per vertex.
template <uint32_t G>
__device__ inline void ms_pull_unit(uint32_t u, uint32_t e, const uint64_t *off, const uint32_t *adj, u64 *vis, u64 *nz1,
                                    uint8_t *bpd, ulonglong2 *bps, const MsLevel &L)
{
    const uint32_t lane = threadIdx.x & 63;
    uint32_t v = 0, deg = 0;
    u64 nu = 0ull, m = 0ull;
    if (u != kEmpty) {
        const uint64_t b = off[u];
        deg = (uint32_t)(off[u + 1] - b);
        if (G < 64 && deg > G) deg = 0;
        nu = L.nxt[u];
        if (e < deg) {
            v = adj[b + e];
            m = L.cur[v] & nu;
        }
    }
    const u64 all = __ballot(m != 0ull);
    for (uint32_t g = 0; g < 64 / G; ++g) {
        // (a vertex put on the level has an edge)
        const uint32_t dg = __builtin_amdgcn_readlane(deg, g * G);
        if (!dg) continue;
        const uint32_t ug = __builtin_amdgcn_readlane(u, g * G);
        const u64 ng = readlane64(nu, g * G);
        const bool on = (ng >> lane) & 1ull, alone = dg <= G;
        if (__builtin_amdgcn_readlane(e, g * G) == 0) {
            if (on) bpd[(uint64_t)ug * kBpdStride + lane] = (uint8_t)(L.d + 1);
            if (lane == 0) vis[ug] |= ng;
        }
        ulonglong2 *r = &bps[(uint64_t)ug * kBP + lane];
        ulonglong2 s = {0ull, 0ull};
        // (a selected neighbour starts with its own bit)
        if (alone && on) s.x = r->x;
        ms_rows(all & group_lanes<G>(g), v, m, [&](const uint32_t (&w)[kMsAhead], const bool (&mine)[kMsAhead]) {
            ulonglong2 y[kMsAhead];
#pragma unroll
            for (uint32_t k = 0; k < kMsAhead; ++k)
                y[k] = mine[k] ? bps[(uint64_t)w[k] * kBP + lane] : make_ulonglong2(0ull, 0ull);
#pragma unroll
            for (uint32_t k = 0; k < kMsAhead; ++k) {
                s.x |= y[k].x;
                s.y |= y[k].y;
            }
        });
        if (alone) {
            if (s.x | s.y) *r = s;
        } else {
            if (s.x) atomicOr(&r->x, s.x);
            if (s.y) atomicOr(&r->y, s.y);
        }
        const u64 nz = __ballot(s.x != 0ull);
        if (lane == 0 && nz) {
            if (alone)
                nz1[ug] |= nz;
            else
                atomicOr(&nz1[ug], nz);
        }
    }
}

// A level's work: the pieces of its larger vertices, then the others four at a
// time.  f64(vertex, edge), f16(vertex, edge) get every lane's.
template <class F64, class F16>
__device__ inline void ms_level_units(const u64 *piece, uint32_t npiece, const uint32_t *list, uint32_t nlist, F64 f64,
                                      F16 f16)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t nw = gridDim.x * (blockDim.x / 64), w = uniform32((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    for (uint32_t c = w; c < npiece; c += nw) {
        const u64 desc = uniform64(piece[c]);
        f64((uint32_t)desc, (uint32_t)(desc >> 32) + lane);
    }
    constexpr uint32_t P = 64 / kMsSmall;
    for (uint32_t c = w * P; c < nlist; c += nw * P) {
        const uint32_t i = c + lane / kMsSmall;
        f16(i < nlist ? list[i] : kEmpty, lane & (kMsSmall - 1));
    }
}

__global__ __launch_bounds__(256) void k_ms_scan(const uint64_t *off, const uint32_t *adj, const u64 *vis,
                                                 const u64 *nz1, ulonglong2 *bps, MsLevel L)
{
    ms_level_units(
        L.cur_piece, L.cnt->piece[L.d][0], L.cur_list, L.cnt->v[L.d][0],
        [&](uint32_t v, uint32_t e) { ms_scan_unit<kMsPiece>(v, e, off, adj, vis, nz1, bps, L); },
        [&](uint32_t v, uint32_t e) { ms_scan_unit<kMsSmall>(v, e, off, adj, vis, nz1, bps, L); });
}

__global__ __launch_bounds__(256) void k_ms_pull(const uint64_t *off, const uint32_t *adj, u64 *vis, u64 *nz1,
                                                 uint8_t *bpd, ulonglong2 *bps, MsLevel L)
{
    ms_level_units(
        L.nxt_piece, L.cnt->piece[L.d + 1][0], L.nxt_list, L.cnt->v[L.d + 1][0],
        [&](uint32_t u, uint32_t e) { ms_pull_unit<kMsPiece>(u, e, off, adj, vis, nz1, bpd, bps, L); },
        [&](uint32_t u, uint32_t e) { ms_pull_unit<kMsSmall>(u, e, off, adj, vis, nz1, bpd, bps, L); });
    if (L.d == 0) return;
    const uint32_t no = L.cnt->v[L.d - 1][0], stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < no; i += stride) L.old[L.old_list[i]] = 0ull;
}

__global__ void k_ms_fill(uint8_t *bpd, uint64_t nbpd, u64 *z0, uint64_t nz0)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint4 *d4 = reinterpret_cast<uint4 *>(bpd);  // (64 bytes per vertex)
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nbpd / 16; i += stride)
        d4[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nz0; i += stride) z0[i] = 0ull;
}

}  // namespace

// Sixteen lanes per vertex: lane l < 13 masks the sets of slots 4l..4l+3 and
// writes their byte of nonempty-set bits, so one pass over the sets (800 B per
// vertex) does both.
__global__ __launch_bounds__(256) void k_bp_finish(uint32_t n, int mask, ulonglong2 *bps, uint8_t *bpd)
{
    const uint32_t l = threadIdx.x & 15u;
    const uint32_t stride = (gridDim.x * blockDim.x) / 16;
    if (l > (kBP - 1) / 4) return;
    for (uint32_t v = (blockIdx.x * blockDim.x + threadIdx.x) / 16; v < n; v += stride) {
        ulonglong2 *row = bps + (uint64_t)v * kBP + 4 * l;
        const uint32_t cnt = min(4u, kBP - 4 * l);
        uint32_t nz = 0;
        for (uint32_t j = 0; j < cnt; ++j) {
            ulonglong2 s = row[j];
            if (mask && (s.x & s.y)) {
                s.y &= ~s.x;
                row[j] = s;
            }
            nz |= (s.x ? 1u << j : 0u) | (s.y ? 16u << j : 0u);
        }
        bpd[(uint64_t)v * kBpdStride + kBpNzByte + l] = (uint8_t)nz;
    }
}

void launch_bp_finish(uint32_t n, bool mask, uint64_t *bps, uint8_t *bpd, hipStream_t st)
{
    hipLaunchKernelGGL(k_bp_finish, dim3(grid_for((uint64_t)n * 16, 256, 16384)), dim3(256), 0, st, n, mask ? 1 : 0,
                       (ulonglong2 *)bps, bpd);
}

void select_bp_roots(uint32_t n, const uint64_t *off, const uint32_t *adj, std::vector<uint8_t> &used,
                     uint32_t *roots, BpSeeds &seeds, const uint32_t *map)
{
    used.assign(n, 0);
    uint32_t r = 0;
    for (uint32_t i = 0; i < kBP; ++i) {
        while (r < n && used[r]) ++r;
        if (r == n) {
            if (roots) roots[i] = kEmpty;
            continue;
        }
        if (roots) roots[i] = r;
        used[r] = 1;
        seeds.v.push_back(map ? map[r] : r);
        seeds.slot.push_back(i);
        seeds.j.push_back(255u);
        const uint64_t deg = off[r + 1] - off[r];
        uint32_t ns = 0;
        for (uint64_t di = 0; di < deg && ns < 64; ++di) {
            const uint32_t v = adj[off[r] + deg - 1 - di];
            if (!used[v]) {
                used[v] = 1;
                seeds.v.push_back(map ? map[v] : v);
                seeds.slot.push_back(i);
                seeds.j.push_back(ns);
                ++ns;
            }
        }
    }
}

pado_gpu_status build_bp_multi(pado_gpu_graph *g, pado_gpu_index *idx, DevBuf<uint8_t> &d_used,
                               std::vector<uint8_t> &h_used)
{
    // Serial root / neighbour selection (PARA:670-709).
    BpSeeds seeds;
    select_bp_roots(g->n, g->h_off.data(), g->h_adj.data(), h_used, idx->bp_roots, seeds, nullptr);
    return build_bp_seeded(g, idx, d_used, h_used, seeds);
}

pado_gpu_status build_bp_seeded(pado_gpu_graph *g, pado_gpu_index *idx, DevBuf<uint8_t> &d_used,
                                const std::vector<uint8_t> &h_used, const BpSeeds &seeds)
{
    hipStream_t st = g->ctx->stream;
    const uint32_t n = g->n;
    const uint64_t m = g->m;
    WorkPool *wp = g->work.get();
    PADO_TRY(idx->bpd.alloc((uint64_t)n * kBpdStride));
    PADO_TRY(idx->bps.alloc((uint64_t)n * kBP * 2));
    PADO_TRY(d_used.alloc(n, wp));
    const std::vector<uint32_t> &sv = seeds.v, &ss = seeds.slot, &sj = seeds.j;
    PADO_HIP(hipMemcpyAsync(d_used.p, h_used.data(), n, hipMemcpyHostToDevice, st));

    // masks[0..2], vis, nz1 (slots with a nonempty S^-1) in one buffer
    DevBuf<u64> masks, pieces[2];
    DevBuf<uint32_t> lists, dseeds;
    DevBuf<MsCounts> cnt;
    PADO_TRY(masks.alloc(5ull * n, wp));
    const uint64_t max_pieces = m / kMsPiece + n;
    PADO_TRY(pieces[0].alloc(max_pieces, wp));
    PADO_TRY(pieces[1].alloc(max_pieces, wp));
    PADO_TRY(lists.alloc(3ull * n, wp));
    PADO_TRY(cnt.alloc(1, wp));
    const uint32_t ns = (uint32_t)sv.size();
    PADO_TRY(dseeds.alloc(3ull * (ns ? ns : 1), wp));
    std::vector<uint32_t> packed(sv);
    packed.insert(packed.end(), ss.begin(), ss.end());
    packed.insert(packed.end(), sj.begin(), sj.end());
    if (ns) PADO_HIP(hipMemcpyAsync(dseeds.p, packed.data(), 4ull * packed.size(), hipMemcpyHostToDevice, st));

    hipLaunchKernelGGL(k_ms_fill, dim3(grid_for((uint64_t)n * kBP, 256, 8192)), dim3(256), 0, st, idx->bpd.p,
                       (uint64_t)n * kBpdStride, (u64 *)idx->bps.p, (uint64_t)n * kBP * 2);
    hipLaunchKernelGGL(k_ms_fill, dim3(grid_for(n, 256, 4096)), dim3(256), 0, st, (uint8_t *)nullptr, 0ull, masks.p,
                       5ull * n);
    hipLaunchKernelGGL(k_ms_fill, dim3(32), dim3(256), 0, st, (uint8_t *)nullptr, 0ull, (u64 *)cnt.p,
                       (uint64_t)sizeof(MsCounts) / 8);

    PinnedBuf<MsCounts> pin;
    PADO_TRY(pin.alloc(wp, st));
    MsCounts *h_cnt = pin.p;
    struct Events {
        hipEvent_t e[2] = {nullptr, nullptr};
        ~Events()
        {
            for (hipEvent_t x : e)
                if (x) (void)hipEventDestroy(x);
        }
    } ev;
    for (hipEvent_t &x : ev.e) PADO_HIP(hipEventCreate(&x));

    ulonglong2 *bps = (ulonglong2 *)idx->bps.p;
    u64 *vis = masks.p + 3ull * n, *nz1 = masks.p + 4ull * n;
    auto level = [&](uint32_t d) {
        auto mask = [&](uint32_t l) { return masks.p + (uint64_t)(l % 3) * n; };
        auto list = [&](uint32_t l) { return lists.p + (uint64_t)(l % 3) * n; };
        return MsLevel{mask(d), mask(d + 1), mask(d + 2),  // (d + 2 = d - 1 mod 3)
                       list(d), list(d + 2), list(d + 1), pieces[d & 1].p, pieces[(d + 1) & 1].p, cnt.p, d};
    };
    // Up to 8,192 resident waves; few for small graphs, whose levels are short.
    // A wave for each piece of a level that has every vertex, at least: with
    // the vertices alone counted, small dense graphs ran on a few compute
    // units (complete graph of 2,000 vertices: 3.8 ms, now 0.3; 16,000 vertices
    // of degree 1,400: 8.1 and 3.6; R-MAT 14: 0.42 and 0.34).
    const uint32_t grid = (uint32_t)std::max<uint64_t>(32u, std::min<uint64_t>(2048u, std::max<uint64_t>(n / 64, m / 256)));
    uint32_t max_level = 0;
    if (ns)
        hipLaunchKernelGGL(k_ms_seed, dim3(grid_for(ns, 256, 4096)), dim3(256), 0, st, ns, dseeds.p, dseeds.p + ns,
                           dseeds.p + 2 * ns, g->off.p, idx->bpd.p, bps, vis, nz1, lists.p, pieces[0].p, level(0));
    // Levels d .. d + block - 1 per host check; the last one ever run is 254
    // (its children would be on level 255, outside the u8 distances).
    uint32_t block = 8;
    for (uint32_t d = 0; ns;) {
        const uint32_t end = std::min<uint32_t>(d + block, kInf8);
        PADO_HIP(hipEventRecord(ev.e[0], st));
        for (; d < end; ++d) {
            const MsLevel L = level(d);
            hipLaunchKernelGGL(k_ms_scan, dim3(grid), dim3(256), 0, st, g->off.p, g->adj.p, vis, nz1, bps, L);
            hipLaunchKernelGGL(k_ms_pull, dim3(grid), dim3(256), 0, st, g->off.p, g->adj.p, vis, nz1, idx->bpd.p, bps,
                               L);
        }
        PADO_HIP(hipEventRecord(ev.e[1], st));
        PADO_HIP(hipMemcpyAsync(h_cnt, cnt.p, sizeof(MsCounts), hipMemcpyDeviceToHost, st));
        PADO_HIP(hipStreamSynchronize(st));
        float ms = 0.f;
        PADO_HIP(hipEventElapsedTime(&ms, ev.e[0], ev.e[1]));
        idx->ktimes.ms_bp += ms;
        while (max_level < end && h_cnt->v[max_level + 1][0]) ++max_level;
        if (max_level < end) break;  // level `end` is empty
        if (max_level >= kInf8) {
            // Wide hop domain: the sweep stops after level 254 (whose sibling
            // sets are complete); vertices farther away keep INF (255) in
            // that slot -- level 255 was written as 255 -- and the labeling
            // and query kernels ignore such slots.
            if (idx->wide) break;
            set_error("bit-parallel BFS reached level 255: graph eccentricity is outside the uint8 "
                      "distance domain of the reference (its level counter wraps at 255)");
            return PADO_GPU_ERR_DOMAIN;
        }
        block = std::min<uint32_t>(2 * block, 64u);
    }
    if (ns) idx->ktimes.n_bp = std::min<uint32_t>(max_level + 1, kInf8);
    launch_bp_finish(n, true, idx->bps.p, idx->bpd.p, st);
    PADO_HIP(hipStreamSynchronize(st));
    idx->bp_max_level = max_level;
    return PADO_GPU_OK;
}

}  // namespace pado
