"""Query kernels at the sizes where their tiles change: label lists around
multiples of a load, a tile and several tiles, against a plain restatement of
query_distance on imported indexes with arbitrary slots, sets and labels, and
batches whose pair counts leave every remainder."""
import ctypes
import struct

import numpy as np
import pytest

import oracle
import parallel_distance_oracle_amd as pado
from helpers import rank_space

pytestmark = pytest.mark.gpu

LENGTHS = (0, 1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 255, 256, 257, 320, 511, 512,
           513, 700)
N = 756  # 27 vertices of each length


def _lists(rng):
    lens = np.array([LENGTHS[i % len(LENGTHS)] for i in range(N)])
    hubs = [np.sort(rng.choice(N, x, replace=False)).astype(np.uint32) for x in lens]
    loff = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    return hubs, loff


def _arbitrary_index(seed, slots):
    """Labels, distances and sets that no graph need have: every combination
    of empty and nonempty sets, unreached slots and equal sums occurs."""
    rng = np.random.default_rng(seed)
    hubs, loff = _lists(rng)
    dist = rng.integers(1, 7, int(loff[-1])).astype(np.uint8)
    bp_d = rng.integers(0, 6, (N, 50)).astype(np.uint8)
    bp_d[rng.random((N, 50)) < (0.3 if slots else 1.0)] = 255
    bits = rng.integers(0, 64, (2, N, 50))
    bp_s = np.where(rng.random((N, 50, 2)) < 0.5, np.uint64(1) << np.moveaxis(bits, 0, 2).astype(np.uint64), 0)
    bp_s[bp_d == 255] = 0
    return bp_d, bp_s.astype(np.uint64), loff, np.concatenate(hubs), dist, hubs


def _expected(ix, a, b, ref_compat):
    bp_d, bp_s, loff, _, dist, hubs = ix
    out = np.empty(a.size, np.uint8)
    td = bp_d[a].astype(np.int64) + bp_d[b]
    xa, ya, xb, yb = bp_s[a, :, 0], bp_s[a, :, 1], bp_s[b, :, 0], bp_s[b, :, 1]
    low = np.where(xa & xb, td - 2, np.where((xa & yb) | (ya & xb), td - 1, td))
    low = np.where((low < 0) | ((td < 2) & ref_compat), 255, low)
    best = low.min(axis=1)
    for i, (p, q) in enumerate(zip(a, b)):
        _, ia, ib = np.intersect1d(hubs[p], hubs[q], assume_unique=True, return_indices=True)
        d = int(best[i])
        if ia.size:
            d = min(d, int((dist[int(loff[p]):][ia].astype(int) + dist[int(loff[q]):][ib]).min()))
        out[i] = 255 if d >= 253 else d
    return out


@pytest.mark.parametrize("slots", (False, True))
def test_list_lengths(gpu_ctx, slots):
    ix = _arbitrary_index(11, slots)
    idx = pado.Index.import_(gpu_ctx, N, *ix[:5])
    order = np.random.default_rng(5).permutation(N).astype(np.uint32)
    idx.order(order)
    # every length against every length
    k = len(LENGTHS)
    a = np.repeat(np.arange(k), k).astype(np.uint32) + k * np.arange(k * k, dtype=np.uint32) % (N - k) // k * k
    b = np.tile(np.arange(k), k).astype(np.uint32) + k * 3
    rng = np.random.default_rng(6)
    a = np.concatenate([a % N, rng.integers(0, N, 3000)]).astype(np.uint32)
    b = np.concatenate([b % N, rng.integers(0, N, 3000)]).astype(np.uint32)
    back = np.argsort(order).astype(np.uint32)
    for ref in (False, True):
        exp = _expected(ix, a, b, ref)
        print(f"[gpu] {a.size} pairs ref={ref} slots={slots}", flush=True)
        assert np.array_equal(idx.query(a, b, ref_compat=ref, rank_space=True), exp)
        assert np.array_equal(idx.query(back[a], back[b], ref_compat=ref), exp)
        one = [idx.query_pair(int(back[x]), int(back[y]), ref_compat=ref) for x, y in zip(a[:300], b[:300])]
        assert np.array_equal(np.array(one, np.uint8), exp[:300])


@pytest.mark.parametrize("count", (1, 2, 3, 5, 63, 64, 65, 255, 257, 70001, 300007))
def test_pair_counts(gpu_ctx, count):
    """Chunks of 4 to 64 pairs per wave and every remainder; some ids lie
    past the index."""
    ix = _arbitrary_index(12, True)
    idx = pado.Index.import_(gpu_ctx, N, *ix[:5])
    idx.order(np.arange(N, dtype=np.uint32))
    rng = np.random.default_rng(count)
    pool_a, pool_b = rng.integers(0, N, 500).astype(np.uint32), rng.integers(0, N, 500).astype(np.uint32)
    exp = _expected(ix, pool_a, pool_b, False)
    pick = rng.integers(0, 500, count)
    a, b, e = pool_a[pick], pool_b[pick], exp[pick]
    far = rng.random(count) < 0.1
    a[far] += N
    e = np.where(far, np.where(a == b, 0, 255), e)
    print(f"[gpu] {count} pairs", flush=True)
    assert np.array_equal(idx.query(a, b), e)


def test_weighted_list_lengths(gpu_ctx, tmp_path):
    rng = np.random.default_rng(21)
    hubs, loff = _lists(rng)
    dist = rng.integers(0, 30000, int(loff[-1]))
    path = tmp_path / "w.index"
    with open(path, "wb") as f:  # the reference's weighted file: u32 hub, i16 distance
        f.write(struct.pack("<I", N))
        for v in range(N):
            f.write(struct.pack("<I", hubs[v].size))
            for h, d in zip(hubs[v], dist[int(loff[v]):int(loff[v + 1])]):
                f.write(struct.pack("<Ih", int(h), int(d)))
    h = ctypes.c_void_p()
    fn = pado.lib().pado_gpu_windex_load
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p)]
    assert fn(gpu_ctx.h, str(path).encode(), ctypes.byref(h)) == 0
    idx = pado.Index(gpu_ctx, h)
    k = len(LENGTHS)
    a = np.concatenate([np.repeat(np.arange(k), k), rng.integers(0, N, 3000)]).astype(np.uint32)
    b = np.concatenate([np.tile(np.arange(k), k) + k * 4, rng.integers(0, N, 3000)]).astype(np.uint32)
    exp = np.full(a.size, pado.WINF, np.uint32)
    for i, (p, q) in enumerate(zip(a, b)):
        _, ia, ib = np.intersect1d(hubs[p], hubs[q], assume_unique=True, return_indices=True)
        if ia.size:
            exp[i] = (dist[int(loff[p]):][ia] + dist[int(loff[q]):][ib]).min()
    print(f"[gpu] {a.size} weighted pairs", flush=True)
    assert np.array_equal(idx.query(a, b), exp)
    assert np.array_equal(idx.query(a, b, ref_compat=True), np.where(exp >= 32765, 32767, exp))
    assert np.array_equal(np.array([idx.query_pair(int(x), int(y)) for x, y in zip(a[:300], b[:300])], np.uint32),
                          exp[:300])


@pytest.mark.parametrize("kind", ("hops", "wide", "cut", "weighted"))
def test_components(gpu_ctx, kind):
    """More components than bit-parallel slots, isolated vertices among them;
    "cut" has a path deeper than the slots' BFS goes."""
    rng = np.random.default_rng(3)
    parts, n = [], 0

    def add(edges, size):
        nonlocal n
        parts.append(np.asarray(edges, np.uint32).reshape(-1, 2) + np.uint32(n))
        n += size

    add(pado.rmat_edges(8, 6, seed=4), 256)
    add(pado.grid_edges(9, 0.1, 2), 81)
    if kind == "cut":
        add([(i, i + 1) for i in range(399)], 400)
    for k in range(120):
        size = 2 + k % 5
        add([(i, i + 1) for i in range(size - 1)], size)
        n += k % 2  # an isolated vertex
    edges = np.concatenate(parts + [np.array([[n, n + 1]], np.uint32)])
    n += 2
    w = pado.edge_weights(edges.shape[0], 1, 100, 5)
    G, rank, _ = rank_space(edges)
    dg, _, _ = pado.DeviceGraph.from_edges(gpu_ctx, edges, w if kind == "weighted" else None, rank)
    idx = pado.Index.build(gpu_ctx, dg, wide=kind in ("wide", "cut"))
    idx.order(rank)
    a, b = rng.integers(0, n, 20000).astype(np.uint32), rng.integers(0, n, 20000).astype(np.uint32)
    a[:n] = b[:n] = np.arange(n)
    if kind == "weighted":
        import scipy.sparse as sp
        from scipy.sparse.csgraph import dijkstra

        e = edges.astype(np.int64)
        A = sp.coo_matrix((w.astype(float), (e[:, 0], e[:, 1])), shape=(n, n)).tocsr()
        d = dijkstra(A, directed=False)[a, b]
        exp = np.where(np.isinf(d), float(pado.WINF), d).astype(np.uint32)
    else:
        hops = oracle.bfs_pairs(G.num_v, G.off, G.adj, rank[a], rank[b])
        exp = oracle.bfs_to_u8(hops) if kind == "hops" else np.minimum(hops, pado.WIDE_INF).astype(np.uint16)
    print(f"[gpu] {kind}: {n} vertices", flush=True)
    assert np.array_equal(idx.query(a, b), exp)
    assert np.array_equal(idx.query(rank[a], rank[b], rank_space=True), exp)

