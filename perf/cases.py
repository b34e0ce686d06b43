"""Performance cases: what users of the framework have it do, at real sizes.

Graphs are R-MAT (a, b, c, d = 0.57, 0.19, 0.19, 0.05, the benchmark's own
parameters) or square grids with 5% of the edges deleted (road-like: deep,
wide hop domain).  Kinds of case:

  pairs   one-pair calls in a loop (the reference driver's query loop)
  host    a batch of pairs in host arrays, answers in a host array
  device  a batch of pairs resident in HBM, answers left in HBM
  serve   a burst of requests through the query server
  build   index of a resident graph, ordered, then a first batch of queries
          (and, on request, its labels exported)
  ingest  edge list -> device graph -> index -> ordered -> exported labels
  multi   many graphs labeled as one job, then queried graph by graph

listed() holds the standing cases, draw() others of the same ranges.
"""
import numpy as np
import torch

# torch first, then the library: the library then runs on the HIP runtime
# that torch has loaded, and both see each other's device memory.
import parallel_distance_oracle_amd as pado

_RECORD_BYTES = 858  # one vertex's bit-parallel record (50 x 17 B) and label offset


def listed():
    return [
        # A driver asking pair by pair, as the reference's own loop does.
        {"name": "pairs_small", "kind": "pairs", "graph": "rmat", "vertices": 16301, "ef": 8, "pairs": 64},
        # A service call with one user's worth of pairs: latency.
        {"name": "host_1k", "kind": "host", "graph": "rmat", "vertices": 65407, "ef": 16, "pairs": 1000},
        # An analytics job whose pairs come from host memory.
        {"name": "host_6m", "kind": "host", "graph": "rmat", "vertices": 261901, "ef": 16, "pairs": 6000001},
        # The benchmark's batch query: uniform pairs over the largest index.
        {"name": "device_10m", "kind": "device", "graph": "rmat", "vertices": 1048291, "ef": 16, "pairs": 10000000},
        # The serving index and its pair mix (half the pairs Zipf over degree rank).
        {"name": "device_zipf", "kind": "device", "graph": "rmat", "vertices": 16301, "ef": 8, "pairs": 1000003,
         "zipf": True},
        # Weighted distances over a social-network-like graph.
        {"name": "device_weighted", "kind": "device", "graph": "rmat", "vertices": 261901, "ef": 16, "pairs": 2000000,
         "weighted": True},
        # The benchmark's request sizes (log-uniform up to 65,536 pairs), sent as one burst.
        {"name": "serve_burst", "kind": "serve", "graph": "rmat", "vertices": 16301, "ef": 8, "requests": 400,
         "zipf": True},
        # A small graph from its edge list to exported labels.
        {"name": "ingest_small", "kind": "ingest", "graph": "rmat", "vertices": 16301, "ef": 8},
        # The benchmark's headline build.
        {"name": "build_20", "kind": "build", "graph": "rmat", "vertices": 1048291, "ef": 16, "pairs": 1000000},
        # A road-like graph deeper than 254 hops, its labels saved.
        {"name": "build_deep", "kind": "build", "graph": "grid", "side": 161, "pairs": 100000,
         "export": True},
        # The weighted build.
        {"name": "build_weighted_20", "kind": "build", "graph": "rmat", "vertices": 1048291, "ef": 16, "pairs": 1000000,
         "weighted": True},
        # Many small graphs in one job, half R-MAT, half grids.
        {"name": "multi_24", "kind": "multi", "graphs": 24, "lo": 10.0, "hi": 13.5, "pairs": 5000},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], uniform over the logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def _rmat(rng, lo, hi):
    """An R-MAT graph of 2^lo to 2^hi vertices."""
    return {"graph": "rmat", "vertices": _log(rng, 1 << lo, 1 << hi), "ef": rng.randint(5, 16)}


def draw(rng):
    kind = rng.choice(["pairs", "host", "host", "device", "device", "device", "serve", "ingest", "build", "build",
                       "multi"])
    if kind == "pairs":
        return {"kind": kind, **_rmat(rng, 10, 18), "pairs": _log(rng, 16, 256), "weighted": rng.random() < 0.3}
    if kind in ("host", "device"):
        pairs = _log(rng, 100, 8000000)
        if rng.random() < 0.2:
            return {"kind": kind, "graph": "grid", "side": rng.randint(24, 160), "pairs": min(pairs, 2000000)}
        weighted = rng.random() < 0.35
        return {"kind": kind, **_rmat(rng, 10, 18 if weighted else 20), "pairs": pairs, "weighted": weighted,
                "zipf": rng.random() < 0.4}
    if kind == "serve":
        return {"kind": kind, **_rmat(rng, 11, 17), "requests": _log(rng, 20, 400), "zipf": rng.random() < 0.7}
    if kind == "ingest":
        return {"kind": kind, **_rmat(rng, 8, 16), "weighted": rng.random() < 0.3}
    if kind == "build":
        if rng.random() < 0.3:
            return {"kind": kind, "graph": "grid", "side": rng.randint(24, 200), "pairs": _log(rng, 1000, 100000),
                    "export": rng.random() < 0.5}
        return {"kind": kind, **_rmat(rng, 11, 19), "pairs": _log(rng, 1000, 1000000),
                "weighted": rng.random() < 0.35}
    return {"kind": kind, "graphs": rng.randint(4, 24), "lo": 10.0, "hi": round(rng.uniform(11.0, 13.5), 2),
            "pairs": _log(rng, 500, 5000)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rmat_edges(n, ef, seed):
    """Undirected R-MAT edges (u < v) among n vertices, self-loops and repeats
    removed; the last vertex always has one."""
    g = _generator(seed)
    scale = (n - 1).bit_length()
    m = ef << scale
    u = torch.zeros(m, dtype=torch.int64, device="cuda")
    v = torch.zeros(m, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        r = torch.rand(m, generator=g, device="cuda")
        u = (u << 1) | (r >= 0.76)
        v = (v << 1) | (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    keep = (u != v) & (u < n) & (v < n)
    key = (torch.minimum(u, v)[keep] << 32) | torch.maximum(u, v)[keep]
    key = torch.unique(torch.cat([key, torch.tensor([n - 1], device="cuda")]))
    edges = torch.stack([key >> 32, key & 0xFFFFFFFF], dim=1).to(torch.int32)
    return edges.cpu().numpy().view(np.uint32)


def _edges(case, seed):
    if case["graph"] == "grid":
        return pado.grid_edges(case["side"], 0.05, seed)
    return _rmat_edges(case["vertices"], case["ef"], seed)


def _weights(case, edges, seed):
    return pado.edge_weights(edges.shape[0], 1, 100, seed) if case.get("weighted") else None


def _wide(case):
    return case["graph"] == "grid"


def _pairs(case, n, count, seed, rank2id=None):
    a, b = pado.uniform_pairs(n, count, seed)
    if case.get("zipf"):
        half = count // 2
        a[half:] = pado.zipf_vertices(n, count - half, 1.1, seed + 1, rank2id)
        b[half:] = pado.zipf_vertices(n, count - half, 1.1, seed + 2, rank2id)
    return a, b


def _graph(case, seed):
    edges = _edges(case, seed)
    return pado.DeviceGraph.from_edges(pado.default_context(), edges, _weights(case, edges, seed))


def _index(case, seed):
    """(ordered index, rank2id) of the case's graph."""
    dg, rank, rank2id = _graph(case, seed)
    idx = pado.Index.build(pado.default_context(), dg, wide=_wide(case))
    idx.order(rank)
    dg.close()
    return idx, rank2id


def _job(case, seed):
    """Graphs of the multi-graph job: vertex counts log-uniform in
    [2^lo, 2^hi], R-MAT (edge factor 8) and holed grids in turn."""
    r = np.random.RandomState(seed % (1 << 31))
    graphs = []
    for i in range(case["graphs"]):
        nv = 2.0 ** r.uniform(case["lo"], case["hi"])
        if i % 2 == 0:
            e = pado.rmat_edges(int(round(np.log2(nv))), 8, seed=seed + i)
        else:
            e = pado.grid_edges(int(round(np.sqrt(nv))), 0.05, seed + i)
        G = pado.Graph.from_edges(e)
        G.id_transfer(G.make_rank())
        graphs.append(G)
    return graphs


def _label_buffers(case, s):
    """The program's own buffers for exported hubs and distances, with room to
    spare over the label counts of these graphs."""
    n = case["side"] ** 2 if s["wide"] else case["vertices"]
    room = n * (200 if case.get("weighted") or s["wide"] else 40)
    s["hub"] = np.zeros(room, np.int32)
    s["dist"] = np.zeros(room, np.int32 if case.get("weighted") else np.int16 if s["wide"] else np.uint8)


def _export(s, idx):
    *rest, hub, dist = idx.wexport() if idx.weighted else idx.export()
    s["hub"][: hub.size] = _signed(hub)
    s["dist"][: hub.size] = _signed(dist)
    return {"rest": [_signed(x) for x in rest], "hub": s["hub"], "dist": s["dist"]}


def prepare(case, seed):
    ctx = pado.default_context()
    kind = case["kind"]
    s = {"kind": kind, "ctx": ctx, "wide": False}
    if kind == "multi":
        s["graphs"] = _job(case, seed)
        s["pairs"] = [pado.uniform_pairs(G.num_v, case["pairs"], seed + i) for i, G in enumerate(s["graphs"])]
        return s
    s["wide"] = _wide(case)
    if kind == "ingest":
        s["edges"] = _edges(case, seed)
        s["weights"] = _weights(case, s["edges"], seed)
        _label_buffers(case, s)
        return s
    if kind == "build":
        s["graph"], s["rank"], rank2id = _graph(case, seed)
        s["a"], s["b"] = _pairs(case, s["graph"].num_v, case["pairs"], seed, rank2id)
        if case.get("export"):
            _label_buffers(case, s)
        return s
    idx, rank2id = _index(case, seed)
    s["index"] = idx
    if kind == "serve":
        k = case["requests"]
        sizes = np.exp((np.random.RandomState(seed % (1 << 31)).permutation(k) + 0.5) / k * np.log(65536))
        s["off"] = np.concatenate([[0], np.cumsum(sizes.astype(np.int64))]).astype(np.uint64)
        s["a"], s["b"] = _pairs(case, idx.num_v, int(s["off"][-1]), seed, rank2id)
        # Each request holds both kinds of pair, as its users' mix does.
        mix = np.random.RandomState((seed + 1) % (1 << 31)).permutation(s["a"].size)
        s["a"], s["b"] = s["a"][mix], s["b"][mix]
        s["arrival"] = np.zeros(case["requests"])
        s["server"] = pado.Server(ctx, idx, staging_pairs=16 << 20, max_launch_pairs=4 << 20, streams=3)
        return s
    s["a"], s["b"] = _pairs(case, idx.num_v, case["pairs"], seed, rank2id)
    if kind == "device":
        s["a"] = torch.from_numpy(s["a"].view(np.int32)).cuda()
        s["b"] = torch.from_numpy(s["b"].view(np.int32)).cuda()
        out = torch.int32 if idx.weighted else torch.int16 if idx.wide else torch.uint8
        s["out"] = torch.empty(case["pairs"], dtype=out, device="cuda")
        torch.cuda.synchronize()
    elif kind == "pairs":
        s["a"], s["b"] = s["a"].tolist(), s["b"].tolist()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "pairs":
        idx = s["index"]
        return np.array([idx.query_pair(a, b) for a, b in zip(s["a"], s["b"])], np.int64)
    if kind == "host":
        return _signed(s["index"].query(s["a"], s["b"]))
    if kind == "device":
        s["index"].query_device(s["a"].data_ptr(), s["b"].data_ptr(), s["a"].numel(), s["out"].data_ptr())
        return s["out"]
    if kind == "serve":
        _, answers, _ = s["server"].replay(s["a"], s["b"], s["off"], s["arrival"])
        return _signed(answers)
    if kind == "build":
        idx = pado.Index.build(s["ctx"], s["graph"], wide=s["wide"])
        idx.order(s["rank"])
        out = {"labels": int(idx.info.num_labels), "answers": _signed(idx.query(s["a"], s["b"]))}
        if "hub" in s:
            out.update(_export(s, idx))
        return out
    if kind == "ingest":
        dg, rank, rank2id = pado.DeviceGraph.from_edges(s["ctx"], s["edges"], s["weights"])
        idx = pado.Index.build(s["ctx"], dg)
        idx.order(rank)
        return {"rank2id": _signed(rank2id), **_export(s, idx)}
    job = pado.MultiIndex(s["ctx"], s["graphs"])
    return [_signed(job.query(g, a, b)) for g, (a, b) in enumerate(s["pairs"])]


def _signed(x):
    """The same bytes as a signed type where torch has no unsigned one."""
    return x if x.dtype == np.uint8 else x.view(f"i{x.dtype.itemsize}")


# ---------------------------------------------------------------------------
# The work of one pass, and exact answers
# ---------------------------------------------------------------------------
def _size(case):
    """(vertices, directed edges, labels), as the generators give them on
    average; label counts interpolate measured ones."""
    if case["graph"] == "grid":
        n = case["side"] ** 2
        return n, 3.8 * n, 0.45 * case["side"] * n
    n = float(case["vertices"])
    scale, m = float(np.log2(n)), 1.9 * case["ef"] * n
    if case.get("weighted"):
        mean = 135.0 * 1.29 ** (scale - 20)  # 141.7M labels at scale 20, 939.8M at 22
    else:
        mean = 80.4 * 1.84 ** (scale - 20)  # 84.3M labels at scale 20, 6.3M at 18, 0.4M at 16
        mean = max(mean, 0.7)
    return n, m, mean * n


def work(case):
    kind = case["kind"]
    if kind == "multi":
        n = case["graphs"] * 2.0 ** ((case["lo"] + case["hi"]) / 2)
        return {"bytes": n * (_RECORD_BYTES + 4 * 10 + 5 * 20) + case["graphs"] * case["pairs"] * 10, "flops": 0}
    n, m, labels = _size(case)
    record = 0 if case.get("weighted") else _RECORD_BYTES - 8
    label = 8 if case.get("weighted") else 5
    answer = 4 if case.get("weighted") else 2 if _wide(case) else 1
    index = n * (record + 8) + label * labels
    graph = 8 * n + (5 if case.get("weighted") else 4) * m
    if kind == "ingest":
        return {"bytes": 4 * m + index, "flops": 0}
    pairs = case["requests"] * 5909.0 if kind == "serve" else float(case["pairs"])
    # A batch reads each record that it touches once: at most the whole index.
    asked = pairs * (8 + answer) + min(index, pairs * 2 * (record + 8 + label * labels / n))
    if kind == "build":
        return {"bytes": graph + index + asked, "flops": 0}
    return {"bytes": asked, "flops": 0}


def exact(case, seed):
    """Distances by relaxing every edge until nothing changes, from every
    source that is asked for; only for graphs where that is quick."""
    if case["kind"] not in ("pairs", "host", "device") or case.get("vertices", 1) > 1 << 16 or case.get("side", 0) > 64:
        return None
    edges = _edges(case, seed)
    w = _weights(case, edges, seed)
    e = torch.from_numpy(edges.astype(np.int64)).cuda()
    n = int(e.max()) + 1
    tail, head = torch.cat([e[:, 0], e[:, 1]]), torch.cat([e[:, 1], e[:, 0]])
    step = torch.ones(head.numel(), dtype=torch.int64, device="cuda")
    if w is not None:
        step = torch.from_numpy(w.astype(np.int64)).cuda().repeat(2)
    s = prepare(case, seed)
    a, b = (torch.as_tensor(s[x].astype(np.int64) if isinstance(s[x], np.ndarray) else s[x]).cuda().long()
            for x in "ab")
    far = 1 << 40
    sources, which = torch.unique(a, return_inverse=True)
    if sources.numel() * head.numel() > 3 << 32:
        return None
    out = torch.empty_like(a)
    chunk = max(1, (1 << 28) // head.numel())
    for c in range(0, sources.numel(), chunk):
        src = sources[c:c + chunk]
        d = torch.full((n, src.numel()), far, dtype=torch.int64, device="cuda")
        d[src, torch.arange(src.numel(), device="cuda")] = 0
        while True:
            new = d.scatter_reduce(0, head[:, None].expand(-1, src.numel()), d[tail] + step[:, None], "amin")
            if torch.equal(new, d):
                break
            d = new
        mine = (which >= c) & (which < c + src.numel())
        out[mine] = d[b[mine], which[mine] - c]
    if case.get("weighted"):
        return torch.where(out >= far, torch.full_like(out, -1), out)
    if _wide(case):
        return torch.where(out >= far, torch.full_like(out, -1), out)
    return torch.where(out >= 253, torch.full_like(out, 255), out)
