"""Temporaries kept per context: builds of several sizes and kinds one after
the other and on two threads of one context give the oracle's labels, idle
memory goes back with the graphs, and a graph may outlive its context."""
import ctypes
import threading

import numpy as np
import pytest

import oracle
import parallel_distance_oracle_amd as pado
from helpers import rank_space

pytestmark = pytest.mark.gpu

SHAPES = ((9, 4), (12, 8), (11, 3), (13, 6))  # R-MAT scale, edges per vertex


def _case(scale, ef):
    edges = pado.rmat_edges(scale, ef, seed=scale)
    G, rank, _ = rank_space(edges)
    rng = np.random.default_rng(scale)
    a, b = rng.integers(0, G.num_v, 2000).astype(np.uint32), rng.integers(0, G.num_v, 2000).astype(np.uint32)
    return edges, rank, a, b, oracle.bfs_to_u8(oracle.bfs_pairs(G.num_v, G.off, G.adj, rank[a], rank[b]))


def _check(ctx, case):
    edges, rank, a, b, exp = case
    dg, _, _ = pado.DeviceGraph.from_edges(ctx, edges, None, rank)
    for wide in (False, True):
        idx = pado.Index.build(ctx, dg, wide=wide)
        idx.order(rank)
        got = idx.query(a, b)
        assert np.array_equal(got, exp if not wide else np.where(exp == 255, pado.WIDE_INF, exp.astype(np.uint16)))
    return dg


def test_sizes_and_threads():
    ctx = pado.Context(0)
    cases = [_case(*s) for s in SHAPES]
    for c in cases + cases[::-1]:
        _check(ctx, c)
    print("[gpu] one thread done", flush=True)
    errors = []

    def work(order):
        try:
            for i in order:
                _check(ctx, cases[i])
        except BaseException as e:  # reported below
            errors.append(e)

    ts = [threading.Thread(target=work, args=(o,)) for o in ((0, 1, 2, 3), (3, 1, 0, 2))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    # (the HIP runtime that the library itself uses)
    assert pado.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_idle_memory_goes_back():
    ctx = pado.Context(0)
    edges = pado.rmat_edges(17, 8, seed=1)
    before = _free_bytes()
    dg, rank, _ = pado.DeviceGraph.from_edges(ctx, edges)
    idx = pado.Index.build(ctx, dg)
    idx.close()
    held = before - _free_bytes()
    print(f"[gpu] held while the graph lives: {held >> 20} MiB", flush=True)
    dg.close()
    # 256 MiB stay at most; as much again for the runtime's own allocations
    assert before - _free_bytes() <= 512 << 20
    dg2, _, _ = pado.DeviceGraph.from_edges(ctx, edges)
    ctx.close()
    dg2.close()  # after its context
