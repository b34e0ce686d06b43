"""Batches of 4,096 roots (four of the reference's at once) against batches of
1,024, and against the oracle, at the vertex counts where a batch, one of its
quarters or the whole scheme begins."""
import numpy as np
import pytest

import oracle
import parallel_distance_oracle_amd as pado
from helpers import rank_space

pytestmark = pytest.mark.gpu

SET_STATS = ("iterations", "pushes", "ind_pass", "bp_pruned", "cands", "dq_pruned", "num_labels", "labels_appended")


def _graph(kind, n):
    """n vertices: R-MAT with a tail of 40 hops, or a strip 12 wide (distances
    far above 128 for the larger n)."""
    if kind == "strip":
        k = np.arange(n - 1)
        e = np.concatenate([np.stack([k, k + 1], 1)[(k + 1) % 12 != 0], np.stack([k[:n - 12], k[:n - 12] + 12], 1)])
        keep = np.random.default_rng(n).random(e.shape[0]) > 0.03
        keep[-1] = True  # the last vertex has an edge
        return e[keep].astype(np.uint32)
    e = pado.rmat_edges(int(n - 1).bit_length(), 6, seed=n).astype(np.int64)
    e = e[(e < n - 40).all(axis=1)]
    t = np.arange(n - 41, n - 1)
    return np.concatenate([e, np.stack([t, t + 1], 1)]).astype(np.uint32)


def _build(ctx, dg, wide, pull_ratio):
    cfg = pado.BuildCfg()
    cfg.flags = pado.BUILD_WIDE if wide else 0
    cfg.pull_ratio = pull_ratio  # given: batches one by one
    idx = pado.Index.build(ctx, dg, cfg=cfg)
    out = idx.export(), {k: idx.stats()[k] for k in SET_STATS}
    idx.close()
    return out


@pytest.mark.parametrize("kind,n", [("rmat", n) for n in (1024, 1025, 2047, 2049, 4095, 4096, 4097, 5121, 9001)]
                         + [("strip", n) for n in (1500, 2040, 4200)])
@pytest.mark.parametrize("wide", (False, True))
def test_rows(gpu_ctx, kind, n, wide):
    G, _, _ = rank_space(_graph(kind, n))
    assert G.num_v == n
    if kind == "strip" and n == 4200:
        if not wide:
            pytest.skip("deeper than 254 hops")
    dg = pado.DeviceGraph(gpu_ctx, G)
    print(f"[gpu] {kind} n={n} wide={wide}", flush=True)
    got, st = _build(gpu_ctx, dg, wide, 0)
    one, st1 = _build(gpu_ctx, dg, wide, 0xFFFFFFFF)
    dg.close()
    assert st == st1
    for x, y in zip(got, one):
        assert np.array_equal(x, y)
    if not wide:
        X = oracle.Index(G.num_v, G.off, G.adj)
        assert np.array_equal(got[2], X.loff) and np.array_equal(got[3], X.hub) and np.array_equal(got[4], X.dist)
        assert st["iterations"] == X.stats["iters"]
