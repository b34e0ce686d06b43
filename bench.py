"""PADO on one MI355X: R-MAT-20 label build seconds, plus query and serving throughput.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--scale 20] [--edge-factor 16]
                    [--pairs 10000000] [--weighted-scale 22] [--multi-graphs 1024]
                    [--no-cpu] [--cpu-scale 18] [--cpu-pairs 2000000] [--cpu-full]

A step is one full index build (pado_gpu_build: 50 bit-parallel BFSes + all
1024-root batches + the canonical sort) of the R-MAT graph, whose rank-space
CSR is already resident in HBM when the timed region starts.  value = mean
build seconds over the K timed steps (lower is better).  The line also carries:
  parity     -- the last build's label / bit-parallel digests against the
                reference digests recorded in tests/golden (R-MAT 20: the
                reference OpenMP build's own output),
  query      -- plain single-batch GPU queries (10M uniform pairs by default),
                HIP-event timed on the query stream, first 100K answers checked
                against the reference's query_distance,
  serving    -- the R-MAT 14 index served under open-loop Poisson load; the
                headline is the highest served rate whose p99 latency meets a
                1 ms objective, beside the plain single-batch rate,
  weighted   -- weighted R-MAT 22 (weights U[1,100]) build, Dijkstra spot
                checks and the same serving measurement,
  multi      -- 1,024 graphs labeled as one job,
  roofline   -- the dominant build kernel's algorithmic bytes per launch over
                its HIP-event launch time, in a build of batches one by one,
  cpu_baseline -- the reference OpenMP build (oracle/_ref) on a bounded sample
                (R-MAT 18, median of 3, physical cores) and its query_distance
                single-threaded and OpenMP, with the GPU time for the same
                sample beside it (--cpu-full: the same on the R-MAT 20 graph).
Progress goes to stderr; the JSON line to stdout.
"""
import argparse
import hashlib
import json
import os
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import parallel_distance_oracle_amd as pado  # noqa: E402

HBM_PEAK_GBS = 8000.0
BP_RECORD_BYTES = 50 * (1 + 8 + 8)  # 850 B: bit-parallel record of one vertex
SERVE_SLO_P99_MS = 1.0  # serving latency objective: p99 of completion - arrival
SERVE_MODE = "launch"  # serving mode of the bench legs (--serve-mode)


def log(*a):
    print("[bench]", *a, file=sys.stderr, flush=True)


def digest(*arrays):
    h = hashlib.sha256()
    for a in arrays:
        h.update(np.ascontiguousarray(a).tobytes())
    return h.hexdigest()


def golden_meta(scale, ef):
    p = os.path.join(ROOT, "tests", "golden", f"rmat{scale}_ef{ef}.json")
    if os.path.exists(p):
        with open(p) as f:
            return json.load(f)
    return None


def make_graph(scale, ef):
    t0 = time.time()
    edges = pado.rmat_edges(scale, ef, 0.57, 0.19, 0.19, 1)
    G = pado.Graph.from_edges(edges)
    rank = G.make_rank()
    rank2id = G.id_transfer(rank)
    log(f"R-MAT {scale} ef{ef}: n={G.num_v} edges={edges.shape[0]} host ingest {time.time() - t0:.1f}s")
    return edges, G, rank, rank2id


def host_cpu():
    """The host's CPU model, sockets x cores, SMT state, and the physical cores
    this process may run on (its affinity set, one logical CPU per core)."""
    info = {"model": None, "sockets": None, "cores_per_socket": None, "threads_per_core": None}
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, check=True).stdout
        for line in out.splitlines():
            k, _, v = line.partition(":")
            v = v.strip()
            if k == "Model name":
                info["model"] = v
            elif k == "Socket(s)":
                info["sockets"] = int(v)
            elif k == "Core(s) per socket":
                info["cores_per_socket"] = int(v)
            elif k == "Thread(s) per core":
                info["threads_per_core"] = int(v)
    except (OSError, subprocess.CalledProcessError, ValueError):
        pass
    aff = sorted(os.sched_getaffinity(0))
    cores = set()
    try:
        out = subprocess.run(["lscpu", "-p=CPU,CORE,SOCKET"], capture_output=True, text=True, check=True).stdout
        for line in out.splitlines():
            if line.startswith("#"):
                continue
            cpu, core, sock = (int(x) if x else 0 for x in line.split(","))
            if cpu in aff:
                cores.add((sock, core))
    except (OSError, subprocess.CalledProcessError, ValueError):
        cores = set(aff)
    info["smt"] = ("on" if (info["threads_per_core"] or 1) > 1 else "off")
    info["affinity_cpus"] = len(aff)
    info["physical_cores_available"] = len(cores) or len(aff)
    return info


def cpu_baseline(ctx, scale, ef, pairs, repeat=3):
    """The reference OpenMP build (oracle/_ref: ParaVertexCentricPLL<1024>
    compiled from the reference's headers) on R-MAT `scale`, `repeat` builds
    (median reported), then its query_distance on `pairs` uniform pairs,
    single-threaded (the reference's own loop, pado.cpp:114-119) and OpenMP
    parallel-for; the GPU build of the same graph timed beside it."""
    import oracle  # noqa: E402  (baseline leg only)

    if not oracle.have_ref():
        return None
    cpu = host_cpu()
    threads = cpu["physical_cores_available"]
    if os.environ.get("OMP_NUM_THREADS"):
        threads = min(threads, int(os.environ["OMP_NUM_THREADS"]))  # this process's CPU share
    edges, G, rank, _ = make_graph(scale, ef)
    dg = pado.DeviceGraph(ctx, G)
    gpu = []
    for _ in range(repeat + 1):
        t0 = time.perf_counter()
        idx = pado.Index.build(ctx, dg)
        ctx.sync()
        gpu.append(time.perf_counter() - t0)
        idx.close()
    dg.close()
    gpu_s = float(np.median(gpu[1:]))
    qa, qb = pado.uniform_pairs(G.num_v, pairs, seed=1)
    log(f"reference build on R-MAT {scale} x{repeat} with {threads} threads, then {pairs} queries ...")
    R = oracle.run_ref(edges, rank, pairs=(qa, qb), threads=threads, repeat=repeat, dump=False,
                       env_extra={"OMP_PROC_BIND": "spread", "OMP_PLACES": "cores"})
    walls = R["build_walls"]
    ref_s = float(np.median(walls))
    log(f"reference R-MAT {scale}: {walls} s (GPU {gpu_s:.3f}s); labeling {R['total_labeling_s']}")
    return {
        "value": round(ref_s, 4), "unit": "s", "cores": threads, "kind": "reference",
        "sample": (f"ParaVertexCentricPLL<1024> build of R-MAT {scale} ef{ef} (n={G.num_v}), constructor wall "
                   f"time, median of {repeat}; OMP_NUM_THREADS={threads} (physical cores available), "
                   f"OMP_PROC_BIND=spread OMP_PLACES=cores; then query_distance on {pairs} uniform pairs"),
        "builds_s": [round(x, 4) for x in walls],
        "total_labeling_time_s": R["total_labeling_s"],
        "gpu_same_sample_s": round(gpu_s, 4),
        "query_pairs": pairs,
        "query_serial_queries_per_s": round(pairs / R["ref_query_serial_s"], 1),
        "query_omp_queries_per_s": round(pairs / R["ref_query_omp_s"], 1),
        "host": cpu,
    }


def serving_leg(ctx, scale=14, ef=8, duration_s=4.0, seed=5, stream=False):
    """The R-MAT 14 index resident; open-loop Poisson arrivals at fixed
    rates; each request carries floor(exp(U(0, ln 65536))) pairs, half
    uniform, half Zipf(1.1) over degree rank.  Latency = completion - arrival
    (admission waits included).  Compared with the plain path: the same pairs
    in one query launch.  stream=True builds the index with per-kernel
    launches and batches one by one (for profiler runs)."""
    edges, G, rank, rank2id = make_graph(scale, ef)
    cfg = pado.BuildCfg()
    cfg.batch_size = pado.BATCH_SIZE
    cfg.flags = pado.BUILD_STREAM if stream else 0
    idx = pado.Index.build(ctx, pado.DeviceGraph(ctx, G), cfg=cfg)
    idx.order(rank)
    res = serve_measure(ctx, idx, G.num_v, rank2id, duration_s, seed)
    res["workload"] = (f"R-MAT {scale} ef{ef} index resident; open-loop Poisson; log-uniform 1..65536 "
                       f"pairs/request; half uniform, half Zipf(1.1) over degree rank")
    return res


def multi_leg(ctx, count, seed=4):
    """Many graphs in one job: `count` graphs with vertex counts log-uniform in
    [2^10, 2^16], half R-MAT (ef 8), half 2D grids with 5% of edges deleted
    (large diameter), labeled by one MultiIndex build: graphs inside the
    reference's u8 domain in interleaved unions, the deep grids on their own in
    the wide hop domain.  Parity (oracle equality, BFS) is checked in
    tests/test_gpu_configs.py on this same workload; here answers from one
    source per graph are spot-checked against a BFS."""
    t0 = time.time()
    graphs = pado.mixed_graphs(count, seed)
    log(f"multi: {count} graphs, {sum(G.num_v for G in graphs)} vertices, host ingest {time.time() - t0:.1f}s")
    times = []
    for rep in range(2):
        t0 = time.perf_counter()
        mi = pado.MultiIndex(ctx, graphs)
        ctx.sync()
        times.append(time.perf_counter() - t0)
        log(f"multi build {rep}: {times[-1]:.3f}s")
        info = mi.info()
        st = [mi.graph_info(g) for g in range(count)]
        if rep == 0:
            mi.close()
    # Spot check: vertex 0 of every 8th graph against a BFS (scipy).
    import scipy.sparse as sp
    from scipy.sparse.csgraph import shortest_path

    spot_ok = True
    for g in range(0, count, 8):
        G = graphs[g]
        n = G.num_v
        rows = np.repeat(np.arange(n), np.diff(G.off.astype(np.int64)))
        A = sp.csr_matrix((np.ones(G.adj.size), (rows, G.adj.astype(np.int64))), shape=(n, n))
        d = shortest_path(A, unweighted=True, indices=0)
        got = mi.query(g, np.zeros(n, np.uint32), np.arange(n, dtype=np.uint32)).astype(np.float64)
        if st[g]["wide"]:
            exp = np.where(np.isinf(d), float(pado.WIDE_INF), d)
        else:
            exp = np.where(np.isinf(d) | (d >= 253), 255.0, d)
        spot_ok &= bool(np.array_equal(got, exp))
    mi.close()
    ok = [x for x in st if x["status"] == 0]
    return {"graphs": count, "vertices": int(sum(G.num_v for G in graphs)),
            "edges": int(sum(int(G.off[-1]) for G in graphs) // 2), "build_s": round(times[-1], 4),
            "graphs_labeled": len(ok), "graphs_wide_domain": sum(1 for x in ok if x["wide"]),
            "graphs_failed": count - len(ok), "labels": int(sum(x["num_labels"] for x in ok)),
            "union_graphs": info["unions"], "bfs_spot_check_ok": spot_ok,
            "workload": "vertex counts log-uniform in [2^10, 2^16]; half R-MAT ef8, half 2D grids with 5% of "
                        "edges deleted; one MultiIndex build (second of two timed)"}


def weighted_build_only(scale, ef=16):
    """Weighted R-MAT build alone (warmup + one timed build), for profiler runs."""
    ctx = pado.Context(0)
    edges = pado.rmat_edges(scale, ef, 0.57, 0.19, 0.19, 1)
    w = pado.edge_weights(edges.shape[0], 1, 100, seed=1)
    G = pado.WeightedGraph.from_edges(edges, w)
    G.id_transfer(G.make_rank())
    dg = pado.DeviceGraph(ctx, G)
    ctx.sync()
    times = []
    for _ in range(2):
        t0 = time.perf_counter()
        idx = pado.Index.build(ctx, dg)
        ctx.sync()
        times.append(time.perf_counter() - t0)
        st = idx.stats()
        idx.close()
    print(json.dumps({"metric": "weighted R-MAT build only (profiling run)", "scale": scale, "value": round(times[-1], 4),
                      "unit": "s", "labels": st["num_labels"], "rounds": st["iterations"]}), flush=True)


def weighted_leg(ctx, scale, ef=16, duration_s=4.0, seed=7, dijkstra_sources=4):
    """Weighted variant: R-MAT `scale` with integer weights U[1,100] from the
    seed, weighted index built and kept resident, served with the same request
    mix; sampled distances checked exact against Dijkstra (scipy)."""
    import scipy.sparse as sp
    from scipy.sparse.csgraph import dijkstra

    t0 = time.time()
    edges = pado.rmat_edges(scale, ef, 0.57, 0.19, 0.19, 1)
    w = pado.edge_weights(edges.shape[0], 1, 100, seed=1)
    G = pado.WeightedGraph.from_edges(edges, w)
    rank = G.make_rank()
    rank2id = G.id_transfer(rank)
    log(f"weighted R-MAT {scale} ef{ef}: n={G.num_v} edges={edges.shape[0]} host ingest {time.time() - t0:.1f}s")
    dg = pado.DeviceGraph(ctx, G)
    ctx.sync()
    t0 = time.perf_counter()
    idx = pado.Index.build(ctx, dg)
    ctx.sync()
    build_s = time.perf_counter() - t0
    st = idx.stats()
    log(f"weighted build {build_s:.3f}s labels={st['num_labels']} rounds={st['iterations']}")
    idx.order(rank)
    # Dijkstra on the original-id graph from a few sources.
    n = G.num_v
    src_rank_space = G.off, G.adj, G.w
    rows = np.repeat(np.arange(n, dtype=np.int64), np.diff(G.off.astype(np.int64)))
    A = sp.csr_matrix((G.w.astype(np.float64), (rows, G.adj.astype(np.int64))), shape=(n, n))
    rng = np.random.default_rng(seed)
    ok = True
    checked = 0
    for s_orig in rng.integers(0, n, dijkstra_sources):
        d = dijkstra(A, directed=False, indices=int(rank[s_orig]), min_only=True)
        tgt = rng.integers(0, n, 20000).astype(np.uint32)
        got = idx.query(np.full(tgt.size, s_orig, np.uint32), tgt).astype(np.float64)
        exp = d[rank[tgt]]
        exp = np.where(np.isinf(exp), float(pado.WINF), exp)
        ok &= bool(np.array_equal(got, exp))
        checked += tgt.size
    del src_rank_space
    res = serve_measure(ctx, idx, n, rank2id, duration_s, seed)
    res.update({"workload": f"weighted R-MAT {scale} ef{ef}, weights U[1,100] seed 1; same request mix",
                "num_v": n, "num_edges": int(edges.shape[0]), "build_s": round(build_s, 4),
                "labels": int(st["num_labels"]), "rounds": int(st["iterations"]),
                "dijkstra_pairs_checked": checked, "dijkstra_exact": ok})
    idx.close()
    dg.close()
    return res


def serve_measure(ctx, idx, n, rank2id, duration_s, seed, max_pairs_per_rate=600_000_000):
    """Open-loop Poisson request stream against a resident ordered index,
    driven by the server's native load generator (pado_gpu_serve_replay)."""
    rng = np.random.default_rng(seed)
    pool_n = 4000
    sizes = np.floor(np.exp(rng.uniform(0, np.log(65536), pool_n))).astype(np.int64)
    sizes = np.maximum(sizes, 1)
    tot = int(sizes.sum())
    ua, ub = pado.uniform_pairs(n, tot, seed=seed)
    za = pado.zipf_vertices(n, tot, 1.1, seed + 1, rank2id)
    zb = pado.zipf_vertices(n, tot, 1.1, seed + 2, rank2id)
    offs = np.concatenate([[0], np.cumsum(sizes)])
    # Request t: first half of its pairs uniform, second half Zipf over degree rank.
    pos = np.arange(tot)
    req_of = np.repeat(np.arange(pool_n), sizes)
    zipf_half = (pos - offs[req_of]) >= (sizes[req_of] // 2)
    allA = np.where(zipf_half, za, ua).astype(np.uint32)
    allB = np.where(zipf_half, zb, ub).astype(np.uint32)
    mean_pairs = tot / pool_n

    # Plain single-batch path on the same pairs (host arrays in and out, one
    # launch); its pageable host copies vary from call to call, so the offered
    # rates are scaled to the best of three calls.
    idx.query(allA[:1000], allB[:1000])
    plain_s = float("inf")
    for _ in range(3):
        t0 = time.perf_counter()
        plain = idx.query(allA, allB)
        plain_s = min(plain_s, time.perf_counter() - t0)
    plain_qps = allA.size / plain_s

    if SERVE_MODE == "resident":
        srv = pado.Server(ctx, idx, staging_pairs=16 << 20, resident=True)
    else:
        srv = pado.Server(ctx, idx, staging_pairs=16 << 20, max_launch_pairs=4 << 20, streams=3)
    # Warm every stream and launch size with a burst of 256 requests, then with
    # a discarded open-loop window (0.25 s at the lowest offered rate): a
    # one-off host stall of several ms has landed in the first open-loop window
    # after a burst.
    srv.replay(allA[:offs[256]], allB[:offs[256]], offs[:257], np.zeros(256))
    w_rate = 0.2 * plain_qps / mean_pairs
    w_m = max(int(w_rate * 0.25), 16)
    w_arr = np.cumsum(rng.exponential(1.0 / w_rate, size=w_m))
    w_off = np.concatenate([[0], np.cumsum(sizes[np.arange(w_m) % pool_n])]).astype(np.uint64)
    w_gather = np.tile(np.arange(tot), -(-w_m // pool_n))[: int(w_off[-1])]
    srv.replay(allA[w_gather], allB[w_gather], w_off, w_arr)
    rates = []
    ok_all = True
    # Offered rates as fractions of the plain batch path; the server overlaps
    # its copies with the label merge, so rates above 1 can still be served.
    for frac in (0.2, 0.4, 0.6, 0.7, 0.8, 0.9, 1.0, 1.2):
        rate_pairs = frac * plain_qps
        rate_req = rate_pairs / mean_pairs
        dur = min(duration_s, max_pairs_per_rate / rate_pairs)
        m = max(int(rate_req * dur), 16)
        arrivals = np.cumsum(rng.exponential(1.0 / rate_req, size=m))
        tmpl = np.arange(m) % pool_n
        ksz = sizes[tmpl]
        roff = np.concatenate([[0], np.cumsum(ksz)]).astype(np.uint64)
        # request i replays template i % pool_n: its pairs follow in order
        gather = np.tile(np.arange(tot), -(-m // pool_n))[: int(roff[-1])]
        A, B = allA[gather], allB[gather]
        lat, ans, wall = srv.replay(A, B, roff, arrivals)
        ok = bool(np.array_equal(ans, plain[gather]))
        ok_all &= ok
        rates.append({"offered_frac_of_plain": frac, "offered_req_per_s": round(rate_req, 1),
                      "offered_queries_per_s": round(rate_pairs, 1), "requests": int(m),
                      "pairs": int(roff[-1]), "window_s": round(float(arrivals[-1]), 4),
                      "served_queries_per_s": round(float(roff[-1]) / wall, 1),
                      "p50_ms": round(float(np.percentile(lat, 50)), 3),
                      "p99_ms": round(float(np.percentile(lat, 99)), 3), "answers_equal_plain": ok})
        log(f"serving {rates[-1]}")
    st = srv.stats()
    srv.stop()
    # Headline: the highest served rate whose p99 latency meets the SLO.
    ok_rates = [r for r in rates if r["p99_ms"] <= SERVE_SLO_P99_MS]
    at_slo = max(ok_rates, key=lambda r: r["served_queries_per_s"]) if ok_rates else None
    sat = max(rates, key=lambda r: r["served_queries_per_s"])
    return {"slo_p99_ms": SERVE_SLO_P99_MS,
            "served_at_slo_queries_per_s": at_slo["served_queries_per_s"] if at_slo else 0.0,
            "p99_ms_at_slo_rate": at_slo["p99_ms"] if at_slo else None,
            "served_at_slo_frac_of_plain": round(at_slo["served_queries_per_s"] / plain_qps, 4) if at_slo else 0.0,
            "plain_batch_queries_per_s": round(plain_qps, 1), "plain_batch_pairs": int(allA.size),
            "rates": rates, "saturation_served_queries_per_s": sat["served_queries_per_s"],
            "p99_ms_at_saturation": sat["p99_ms"], "results_equal_plain_batch": ok_all,
            "launches": st["launches"], "requests": st["requests_done"], "rejected": st["rejected"],
            "busy_ms": round(st["busy_ms"], 2), "mode": SERVE_MODE}


def copy_calibrate(mib):
    """A plain copy of known size: under rocprofv3 --pmc its FETCH_SIZE and
    WRITE_SIZE per dispatch give the counters' scale (expected mib MiB each)."""
    from parallel_distance_oracle_amd.hip import DeviceArray

    n = mib << 20
    ctx = pado.Context(0)
    src = DeviceArray.from_numpy(np.ones(n, np.uint8))
    dst = DeviceArray(n, np.uint8)
    for _ in range(5):
        pado.copy_bytes(ctx, dst.ptr, src.ptr, n)
    ctx.sync()
    assert np.array_equal(dst.numpy()[:4096], np.ones(4096, np.uint8))
    log(f"copied {mib} MiB x 5 with k_copy_bytes")


def load_traffic():
    """HBM bytes per launch of the dominant kernel from the committed PMC
    summary (two rocprofv3 --pmc runs, FETCH_SIZE then WRITE_SIZE, scaled by
    the copy-kernel calibration), or None."""
    p = os.path.join(ROOT, "profiles", "pmc_traffic.json")
    if not os.path.exists(p):
        return None
    with open(p) as f:
        return json.load(f)


ROOFLINE_SCHEDULE = "batches of 1,024 roots one by one"  # of a stream-mode build


def build_roofline(st, timing, traffic, workload):
    """The dominant labeling kernel's algorithmic bytes per launch over its
    launch time.  st: the stats of ONE build, whose launches were timed; what
    they scanned depends on the schedule, so times and counts of different
    builds do not go together.  traffic: load_traffic()."""
    push_bytes = 8 * st["actives"] + 4 * st["edges"] + BP_RECORD_BYTES * st["tails"]
    add_bytes = 5 * st["dq_labels"] + 5 * st["labels_appended"]
    kern = {
        "k_push": (st["ms_push"], st["n_push"], push_bytes),
        "k_add": (st["ms_add"], st["n_add"], add_bytes),
    }
    dom = max(kern, key=lambda k: kern[k][0])
    ms_tot, n_launch, bytes_tot = kern[dom]
    avg_ms = ms_tot / max(n_launch, 1)
    achieved = (bytes_tot / max(n_launch, 1)) / (avg_ms * 1e-3) / 1e9 if avg_ms > 0 else 0.0
    roofline = {"bound": "hbm", "kernel": dom, "achieved": round(achieved, 2), "peak": HBM_PEAK_GBS,
                "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 5), "traffic": None,
                "avg_launch_us": round(avg_ms * 1e3, 2), "launches": int(n_launch),
                "alg_bytes_per_launch": round(bytes_tot / max(n_launch, 1), 1),
                "kernel_ms": {k: round(v[0], 2) for k, v in kern.items()}, "schedule": ROOFLINE_SCHEDULE,
                "timing": timing}
    if traffic and traffic.get("workload") == workload and dom in traffic.get("kernels", {}):
        roofline["traffic"] = traffic["kernels"][dom]["bytes_per_launch"]
        roofline["traffic_source"] = traffic.get("source")
    return roofline


QUERY_RECORD_BYTES = 128  # a vertex's line of the query copy
QUERY_TAIL_BYTES = 16     # its last four words: component, label list


def query_bytes(connected, la, lb):
    """Bytes that a batch of pairs cannot do without: ids and answers, the tail
    of each end's record and, for a connected pair, the two records and label
    lists (la, lb labels).  The set pairs that decide a slot come on top."""
    connected = np.asarray(connected, bool)
    own = 2 * QUERY_RECORD_BYTES + 4 * (np.asarray(la, np.int64) + np.asarray(lb, np.int64))
    return int(np.where(connected, own, 2 * QUERY_TAIL_BYTES).sum()) + 9 * connected.size


def main():
    global SERVE_MODE
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--scale", type=int, default=20)
    ap.add_argument("--edge-factor", type=int, default=16)
    ap.add_argument("--pairs", type=int, default=10_000_000)
    ap.add_argument("--cpu-scale", type=int, default=18,
                    help="R-MAT scale of the bounded CPU-baseline sample (reference OpenMP build)")
    ap.add_argument("--cpu-pairs", type=int, default=2_000_000,
                    help="uniform pairs of the CPU-baseline query leg")
    ap.add_argument("--cpu-full", action="store_true",
                    help="only run the reference OpenMP baseline on the full R-MAT --scale graph (3 builds, "
                         "--pairs queries) with the GPU build beside it, print it and exit")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-serve", action="store_true")
    ap.add_argument("--build-only", action="store_true",
                    help="timed builds and the roofline only (for profiler runs)")
    ap.add_argument("--copy-calibrate", type=int, default=0, metavar="MIB",
                    help="only run a plain device copy of MIB MiB (PMC byte-counter calibration) and exit")
    ap.add_argument("--stream", action="store_true",
                    help="run batches one by one with HIP-event timing of each launch instead of four at a time")
    ap.add_argument("--weighted-scale", type=int, default=22,
                    help="also build and serve a weighted R-MAT of this scale (0 = skip)")
    ap.add_argument("--multi-graphs", type=int, default=1024, metavar="N",
                    help="also label N independent graphs in one job (multi-graph workload; 0 = skip)")
    ap.add_argument("--multi-only", action="store_true", help="only run the multi-graph job and exit")
    ap.add_argument("--weighted-build-only", type=int, default=0, metavar="SCALE",
                    help="only build the weighted R-MAT of this scale (twice: warmup + timed) and exit (profiler runs)")
    ap.add_argument("--serve-mode", choices=("resident", "launch"), default="launch",
                    help="serving with the resident kernel or with one launch per coalesced batch")
    ap.add_argument("--serve-only", action="store_true",
                    help="only run the serving leg and exit (profiler runs; add --stream to build its index "
                         "with per-kernel launches)")
    args = ap.parse_args()
    SERVE_MODE = args.serve_mode
    if args.copy_calibrate:
        copy_calibrate(args.copy_calibrate)
        return
    if args.weighted_build_only:
        weighted_build_only(args.weighted_build_only)
        return
    if args.serve_only:
        res = serving_leg(pado.Context(0), stream=args.stream)
        print(json.dumps({"metric": "serving leg only (profiling run)", "serving": res}), flush=True)
        return
    if args.multi_only:
        print(json.dumps({"metric": "multi-graph labeling job",
                          "multi": multi_leg(pado.Context(0), args.multi_graphs)}), flush=True)
        return
    if args.cpu_full:
        res = cpu_baseline(pado.Context(0), args.scale, args.edge_factor, args.pairs)
        print(json.dumps({"metric": "reference OpenMP baseline, full graph", "cpu_baseline": res}), flush=True)
        return
    if args.gpus != 1:
        print(f"bench.py measures one GPU only; --gpus {args.gpus} is not supported (the index build and "
              f"queries run on a single MI355X)", file=sys.stderr)
        sys.exit(2)
    if pado.device_count() < 1:
        sys.exit("no GPU visible")

    edges, G, rank, rank2id = make_graph(args.scale, args.edge_factor)
    ctx = pado.Context(0)
    dg = pado.DeviceGraph(ctx, G)
    ctx.sync()
    cfg = pado.BuildCfg()
    cfg.batch_size = pado.BATCH_SIZE
    cfg.flags = pado.BUILD_STREAM if args.stream else 0

    for w in range(args.warmup):
        t0 = time.time()
        idx = pado.Index.build(ctx, dg, cfg=cfg)
        ctx.sync()
        log(f"warmup build {w}: {time.time() - t0:.3f}s labels={idx.info.num_labels}")
        idx.close()

    times = []
    idx = None
    ctx.sync()
    for s in range(args.steps):
        if idx is not None:
            idx.close()
        t0 = time.perf_counter()
        idx = pado.Index.build(ctx, dg, cfg=cfg)
        ctx.sync()
        dt = time.perf_counter() - t0
        times.append(dt)
        log(f"build {s}: {dt:.3f}s")
    build_s = float(np.mean(times))
    st = idx.stats()
    log(f"stats: {json.dumps({k: (round(v, 3) if isinstance(v, float) else v) for k, v in st.items()})}")

    # Parity of the last build against the reference digests.
    bp_d, bp_s, loff, hub, dist = idx.export()
    meta = golden_meta(args.scale, args.edge_factor)
    parity = {"labels": int(hub.size)}
    if meta:
        parity["labels_match_reference"] = digest(loff.astype(np.uint64), hub.astype(np.uint32),
                                                  dist.astype(np.uint8)) == meta["labels_sha256"]
        parity["bp_match_reference"] = digest(bp_d.astype(np.uint8), bp_s.astype(np.uint64)) == meta["bp_sha256"]
        parity["bp_hit_count_match_reference"] = st["bp_pruned"] == meta["bp_hit_count"]
        parity["reference_build_s_container"] = meta.get("ref_build_s")
    del bp_d, bp_s, hub, dist

    # Roofline of the dominant labeling kernel (push or add), per launch, from
    # one build of its own: a stream-mode build (a batch at a time) brackets
    # each push / add launch with HIP events on the build stream, which a
    # default build does not, and what it scans is what those launches did.
    timing_src = "timed builds (HIP events on the build stream)"
    st_t = st
    if not args.stream:
        tcfg = pado.BuildCfg()
        tcfg.batch_size = pado.BATCH_SIZE
        tcfg.flags = pado.BUILD_STREAM
        tb = pado.Index.build(ctx, dg, cfg=tcfg)
        ctx.sync()
        st_t = tb.stats()
        tb.close()
        timing_src = "one stream-mode build after the timed builds (HIP events on the build stream)"
    roofline = build_roofline(st_t, timing_src, load_traffic(), f"rmat{args.scale}_ef{args.edge_factor}")
    if args.build_only:
        print(json.dumps({"metric": "R-MAT build only (profiling run)", "value": round(build_s, 4), "unit": "s",
                          "roofline": roofline, "parity": parity, "stats": st, "roofline_stats": st_t}), flush=True)
        return

    # Plain batch query: order by original id, k pairs on device, one launch.
    idx.order(rank)
    qa, qb = pado.uniform_pairs(G.num_v, args.pairs, seed=1)
    query = None
    # Pairs in HBM as buffers of the library's own HIP runtime; one launch of
    # the query kernel on the context's stream, bracketed by HIP events there.
    from parallel_distance_oracle_amd.hip import DeviceArray, Events

    da, db = DeviceArray.from_numpy(qa), DeviceArray.from_numpy(qb)
    out = DeviceArray(args.pairs, np.uint8)
    ev = Events()
    e0, e1 = ev.event(), ev.event()
    stream = ctx.stream
    idx.query_device(da.ptr, db.ptr, args.pairs, out.ptr, stream=stream)
    ctx.sync()
    qt = []
    for _ in range(max(args.steps, 1)):
        ev.record(e0, stream)
        idx.query_device(da.ptr, db.ptr, args.pairs, out.ptr, stream=stream)
        ev.record(e1, stream)
        qt.append(ev.elapsed_ms(e0, e1))
    ev.close()
    q_ms = float(np.mean(qt))
    res = out.numpy()
    da.free()
    db.free()
    out.free()
    query = {"pairs": args.pairs, "ms": round(q_ms, 3), "queries_per_s": round(args.pairs / (q_ms * 1e-3), 1)}
    # Signed (exact) answers must equal the reference's except on its defect set.
    k = min(100_000, args.pairs)
    ref_mode = idx.query(qa[:k], qb[:k], ref_compat=True)
    query["ref_compat_first_100k_match_reference"] = (meta is not None and k == meta["n_pairs"] and
                                                      digest(ref_mode) == meta["answers_sha256"])
    query["exact_vs_ref_compat_differ"] = int(np.count_nonzero(ref_mode != res[:k]))
    lab_per_v = np.diff(loff.astype(np.int64))
    query["alg_bytes"] = query_bytes(res != 255, lab_per_v[rank[qa]], lab_per_v[rank[qb]])
    query["achieved_GBps"] = round(query["alg_bytes"] / (q_ms * 1e-3) / 1e9, 1)
    # The drop-in's query_distance(a, b) loop (pado.cpp:114-119 calls it once
    # per pair): one-pair calls (pado_gpu_query_pair), and the same pairs as
    # one-element batch calls, each checked against the batch answers.
    npair = 2000
    t0 = time.perf_counter()
    one = [idx.query_pair(int(x), int(y)) for x, y in zip(qa[:npair], qb[:npair])]
    t_pair = time.perf_counter() - t0
    t0 = time.perf_counter()
    batch1 = [int(idx.query(qa[i:i + 1], qb[i:i + 1])[0]) for i in range(npair)]
    t_batch1 = time.perf_counter() - t0
    query["pair_calls_us"] = round(t_pair / npair * 1e6, 2)
    query["one_pair_batch_calls_us"] = round(t_batch1 / npair * 1e6, 2)
    query["pair_calls_equal_batch"] = bool(np.array_equal(np.array(one, np.uint8), res[:npair]) and
                                           np.array_equal(np.array(batch1, np.uint8), res[:npair]))
    log(f"query: {query}")

    serving = None
    if not args.no_serve:
        try:
            serving = serving_leg(ctx)
        except Exception as e:
            log(f"serving leg failed: {e}")

    weighted = None
    if args.weighted_scale:
        try:
            weighted = weighted_leg(ctx, args.weighted_scale)
            log(f"weighted: {weighted}")
        except Exception as e:
            log(f"weighted leg failed: {e}")

    multi = None
    if args.multi_graphs:
        try:
            multi = multi_leg(ctx, args.multi_graphs)
            log(f"multi: {multi}")
        except Exception as e:
            log(f"multi-graph leg failed: {e}")

    cpu = None
    if not args.no_cpu:
        try:
            cpu = cpu_baseline(ctx, args.cpu_scale, args.edge_factor, args.cpu_pairs)
        except Exception as e:  # the baseline is reported, never required
            log(f"cpu baseline failed: {e}")

    line = {
        "metric": "R-MAT-20 label build s; served queries/s at p99 latency vs plain batch query",
        "value": round(build_s, 4), "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(build_s * 1e3, 2), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "u8", "data": "synthetic",
        "config": {"workload": f"R-MAT scale {args.scale} ef {args.edge_factor} (0.57,0.19,0.19,0.05) seed 1, "
                               f"BATCH_SIZE=1024, BITPARALLEL_SIZE=50; full index build",
                   "num_v": G.num_v, "num_edges": int(edges.shape[0]),
                   "batch_step": "stream (launch-ahead blocks)" if args.stream else "four batches at a time"},
        "parity": parity, "query": query, "serving": serving, "weighted": weighted, "multi": multi,
        "roofline": roofline, "cpu_baseline": cpu,
        "build_breakdown_ms": {"bp": round(st["ms_bp"], 1), "batches_and_sort": round(st["ms_batch"], 1)},
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
