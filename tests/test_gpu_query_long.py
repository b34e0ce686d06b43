"""Pairs with long label lists: lists around the tiles of a whole wave, in calls
short enough for a wave per pair, in longer ones where groups and whole waves
share the pairs, and around the pair counts where the split changes."""
import ctypes
import struct

import numpy as np
import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu

LENGTHS = (1, 64, 65, 128, 129, 192, 193, 256, 257, 511, 513, 768, 769, 1023, 1024, 1025, 1280, 2047, 2049, 2300)
N = 2400
COUNTS = (4096, 4097, 8192, 8193, 32768, 32769)


def _lists(rng):
    lens = np.array([LENGTHS[i % len(LENGTHS)] for i in range(N)])
    hubs = [np.sort(rng.choice(N, x, replace=False)).astype(np.uint32) for x in lens]
    return hubs, np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)


def _pairs(rng, count):
    k = len(LENGTHS)
    a, b = rng.integers(0, N, count), rng.integers(0, N, count)
    a[:k * k], b[:k * k] = np.repeat(np.arange(k), k), np.tile(np.arange(k), k) + 2 * k
    return a.astype(np.uint32), b.astype(np.uint32)


def _least(hubs, loff, dist, a, b, far):
    """The least sum over common hubs, by a row of distances per first vertex."""
    out = np.full(a.size, far, np.int64)
    row = np.empty(N, np.int64)
    for p in np.unique(a):
        row[:] = far
        row[hubs[p]] = dist[int(loff[p]):int(loff[p + 1])]
        for i in np.flatnonzero(a == p):
            q = b[i]
            out[i] = min(far, int((row[hubs[q]] + dist[int(loff[q]):int(loff[q + 1])]).min()))
    return out


@pytest.fixture(scope="module")
def hops(gpu_ctx):
    rng = np.random.default_rng(31)
    hubs, loff = _lists(rng)
    dist = rng.integers(1, 120, int(loff[-1])).astype(np.uint8)
    bp_d = np.full((N, 50), 255, np.uint8)
    idx = pado.Index.import_(gpu_ctx, N, bp_d, np.zeros((N, 50, 2), np.uint64), loff, np.concatenate(hubs), dist)
    idx.order(np.arange(N, dtype=np.uint32))
    a, b = _pairs(rng, max(COUNTS))
    d = _least(hubs, loff, dist.astype(np.int64), a, b, 255)
    return idx, a, b, np.where(d >= 253, 255, d).astype(np.uint8)


@pytest.mark.parametrize("count", COUNTS)
def test_hops(hops, count):
    idx, a, b, exp = hops
    print(f"[gpu] {count} pairs", flush=True)
    assert np.array_equal(idx.query(a[:count], b[:count]), exp[:count])
    assert np.array_equal(idx.query(a[:count], b[:count], rank_space=True), exp[:count])


@pytest.fixture(scope="module")
def weights(gpu_ctx, tmp_path_factory):
    rng = np.random.default_rng(32)
    hubs, loff = _lists(rng)
    dist = rng.integers(0, 30000, int(loff[-1]))
    path = tmp_path_factory.mktemp("w") / "w.index"
    rec = np.empty(int(loff[-1]), np.dtype([("h", "<u4"), ("d", "<i2")]))
    rec["h"], rec["d"] = np.concatenate(hubs), dist
    with open(path, "wb") as f:  # the reference's weighted file: u32 hub, i16 distance
        f.write(struct.pack("<I", N))
        for v in range(N):
            f.write(struct.pack("<I", hubs[v].size))
            f.write(rec[int(loff[v]):int(loff[v + 1])].tobytes())
    h = ctypes.c_void_p()
    fn = pado.lib().pado_gpu_windex_load
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p)]
    assert fn(gpu_ctx.h, str(path).encode(), ctypes.byref(h)) == 0
    a, b = _pairs(rng, max(COUNTS))
    return pado.Index(gpu_ctx, h), a, b, _least(hubs, loff, dist, a, b, pado.WINF).astype(np.uint32)


@pytest.mark.parametrize("count", COUNTS)
def test_weighted(weights, count):
    idx, a, b, exp = weights
    print(f"[gpu] {count} weighted pairs", flush=True)
    assert np.array_equal(idx.query(a[:count], b[:count]), exp[:count])
