"""Batch calls around the pair counts where the split between groups and whole
waves changes, for indexes on either side of the mean list lengths where it
does (64 and 256), ordered and in rank space, and through the server's
persistent kernel."""
import ctypes
import struct

import numpy as np
import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu

N = 1500
MEANS = (40, 63, 64, 255, 256, 400)
COUNTS = (4095, 4096, 4097, 12288, 12289, 32768, 32769, 65536, 65537, 131073)


def _lists(rng, mean):
    """Lists of 1 to 2 mean - 1 labels, their mean exactly `mean`."""
    lens = rng.integers(1, 2 * mean, N)
    lens[N // 2:] = 2 * mean - lens[:N // 2]
    hubs = [np.sort(rng.choice(N, x, replace=False)).astype(np.uint32) for x in lens]
    return hubs, np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)


def _answers(hubs, loff, dist, a, b, far):
    """All pairs of first vertices a and second ones b: the least sums over common hubs."""
    M = np.full((N, N), far, np.int64)
    for v in range(N):
        M[v, hubs[v]] = dist[int(loff[v]):int(loff[v + 1])]
    out = np.full((a.size, b.size), far, np.int64)
    for i, x in enumerate(a):
        s = M[x][None, hubs[x]] + M[b][:, hubs[x]]
        out[i] = np.minimum(far, s.min(axis=1))
    return out


@pytest.mark.parametrize("mean", MEANS)
@pytest.mark.parametrize("weighted", (False, True))
def test_pair_counts_by_mean_length(gpu_ctx, tmp_path, mean, weighted):
    rng = np.random.default_rng(mean)
    hubs, loff = _lists(rng, mean)
    assert int(loff[-1]) // N == mean
    far = pado.WINF if weighted else 255
    dist = rng.integers(0 if weighted else 1, 30000 if weighted else 120, int(loff[-1]))
    if weighted:
        rec = np.empty(int(loff[-1]), np.dtype([("h", "<u4"), ("d", "<i2")]))
        rec["h"], rec["d"] = np.concatenate(hubs), dist
        path = tmp_path / "w.index"
        with open(path, "wb") as f:  # the reference's weighted file: u32 hub, i16 distance
            f.write(struct.pack("<I", N))
            for v in range(N):
                f.write(struct.pack("<I", hubs[v].size) + rec[int(loff[v]):int(loff[v + 1])].tobytes())
        h = ctypes.c_void_p()
        fn = pado.lib().pado_gpu_windex_load
        fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p)]
        assert fn(gpu_ctx.h, str(path).encode(), ctypes.byref(h)) == 0
        idx = pado.Index(gpu_ctx, h)
    else:
        idx = pado.Index.import_(gpu_ctx, N, np.full((N, 50), 255, np.uint8), np.zeros((N, 50, 2), np.uint64), loff,
                                 np.concatenate(hubs), dist.astype(np.uint8))
        idx.order(np.arange(N, dtype=np.uint32))
    first = rng.choice(N, 200, replace=False)
    second = np.arange(N)
    table = _answers(hubs, loff, dist, first, second, far)
    if not weighted:
        table = np.where(table >= 253, 255, table)
    i, b = rng.integers(0, first.size, max(COUNTS)), rng.integers(0, N, max(COUNTS))
    a, exp = first[i].astype(np.uint32), table[i, b].astype(np.uint32)
    b = b.astype(np.uint32)
    print(f"[gpu] mean {mean} weighted={weighted}", flush=True)
    for k in COUNTS:
        assert np.array_equal(idx.query(a[:k], b[:k]), exp[:k]), k
        if not weighted:  # (a loaded index has no rank-space labels)
            assert np.array_equal(idx.query(a[:k], b[:k], rank_space=True), exp[:k]), k
    srv = pado.Server(gpu_ctx, idx, persistent=True)
    try:
        for k in (3, 5000):
            got, _ = srv.wait(srv.submit(a[:k], b[:k]), k)
            assert np.array_equal(got, exp[:k])
    finally:
        srv.stop()
    idx.close()
