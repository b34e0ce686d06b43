"""A loaded index has the query copy only: calls that need rank-space labels
are refused with a status (no kernel is launched), queries by original id are
answered; files with lists that no record can hold are refused."""
import ctypes
import struct

import numpy as np
import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu

N = 4
STATE, IO = 5, 6


def _load(ctx, fn, path):
    h = ctypes.c_void_p()
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p)]
    return fn(ctx.h, str(path).encode(), ctypes.byref(h)), h


def _weighted_file(path):
    """Vertex x: hub 0 at distance 10 x, and hub x at 0."""
    with open(path, "wb") as f:
        f.write(struct.pack("<I", N))
        for x in range(N):
            labels = [(0, 10 * x)] + ([(x, 0)] if x else [])
            f.write(struct.pack("<I", len(labels)) + b"".join(struct.pack("<Ih", *l) for l in labels))


def _hops_file(path):
    """Vertex x: hub 0 at distance x, and hub x at 0; no bit-parallel labels."""
    with open(path, "wb") as f:
        f.write(struct.pack("<II", N, 50))
        for x in range(N):
            f.write(struct.pack("<BQQ", 255, 0, 0) * 50)
            labels = [(0, x)] + ([(x, 0)] if x else [])
            f.write(struct.pack("<I", len(labels)) + b"".join(struct.pack("<IB", *l) for l in labels))


@pytest.mark.parametrize("weighted", (False, True))
def test_rank_space_calls_are_refused(gpu_ctx, tmp_path, weighted):
    L = pado.lib()
    path = tmp_path / "index"
    (_weighted_file if weighted else _hops_file)(path)
    st, h = _load(gpu_ctx, L.pado_gpu_windex_load if weighted else L.pado_gpu_index_load, path)
    assert st == 0
    idx = pado.Index(gpu_ctx, h)
    a = np.arange(N, dtype=np.uint32)
    exp = a * (10 if weighted else 1)
    assert np.array_equal(idx.query(a, np.zeros(N, np.uint32)), exp)
    out = np.zeros(N, np.uint32 if weighted else np.uint8)
    query = L.pado_gpu_wquery if weighted else L.pado_gpu_query
    for k in (N, 0):
        for flags in (pado.QUERY_RANK_SPACE, pado.QUERY_RANK_SPACE | pado.QUERY_DEVICE_PTRS):
            assert query(gpu_ctx.h, idx.h, pado._p(a), pado._p(a), k, pado._p(out), flags, None) == STATE
    one = ctypes.c_uint32()
    assert L.pado_gpu_query_pair(gpu_ctx.h, idx.h, 0, 1, pado.QUERY_RANK_SPACE, ctypes.byref(one)) == STATE
    off = np.zeros(N + 1, np.uint64)
    if weighted:
        assert L.pado_gpu_windex_export(gpu_ctx.h, idx.h, pado._p(off), None, None) == STATE
    else:
        assert L.pado_gpu_index_export(gpu_ctx.h, idx.h, None, None, pado._p(off), None, None) == STATE
    assert L.pado_gpu_index_order(gpu_ctx.h, idx.h, pado._p(a), N) == STATE
    assert np.array_equal(idx.query(a, np.zeros(N, np.uint32)), exp)
    idx.close()


def test_ordering_that_fails_early_leaves_the_copy():
    ctx = pado.Context(0)
    dg, rank, _ = pado.DeviceGraph.from_edges(ctx, pado.rmat_edges(10, 4, seed=1))
    idx = pado.Index.build(ctx, dg)
    idx.order(rank)
    a, b = pado.uniform_pairs(dg.num_v, 1000, seed=1)
    exp = idx.query(a, b)
    ctx.set_work_limit(1)
    with pytest.raises(pado.PadoError):
        idx.order(rank)
    assert idx.get_info().ordered == 1 and np.array_equal(idx.query(a, b), exp)
    ctx.set_work_limit(0)
    idx.order(rank)
    assert np.array_equal(idx.query(a, b), exp)
    idx.close()
    dg.close()
    ctx.close()


def test_list_longer_than_a_record_holds(gpu_ctx, tmp_path):
    """2^24 labels at one vertex (duplicate hubs, or they would not exist): the
    record's 24-bit count would read as none, and move the list's start."""
    path = tmp_path / "long"
    with open(path, "wb") as f:
        f.write(struct.pack("<II", 1, 1 << 24))
        f.write(bytes(6 << 24))
    assert _load(gpu_ctx, pado.lib().pado_gpu_windex_load, path)[0] == IO
    with open(path, "wb") as f:
        f.write(struct.pack("<II", 1, 1000) + bytes(6000))  # (duplicates alone are taken, as ever)
    st, h = _load(gpu_ctx, pado.lib().pado_gpu_windex_load, path)
    assert st == 0
    idx = pado.Index(gpu_ctx, h)
    assert idx.query([0], [0])[0] == 0
    idx.close()
