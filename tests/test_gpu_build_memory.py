"""Builds in less temporary memory than batches of 4,096 roots take: where
those do not fit, at the start or only when the root-distance table grows, the
build goes on in batches of 1,024, with the same labels; where these do not fit
either it ends with PADO_GPU_ERR_NOMEM."""
import numpy as np
import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def _build(ctx, dg, wide, pull_ratio=0):
    cfg = pado.BuildCfg()
    cfg.flags = pado.BUILD_WIDE if wide else 0
    cfg.pull_ratio = pull_ratio  # given: batches one by one
    idx = pado.Index.build(ctx, dg, cfg=cfg)
    out = idx.export()
    idx.close()
    return out


@pytest.mark.parametrize("wide", (False, True))
def test_smaller_batches_where_the_wide_rows_do_not_fit(wide):
    ctx = pado.Context(0)
    # (above 2^16 vertices, so that the root-distance table grows during the build)
    dg, _, _ = pado.DeviceGraph.from_edges(ctx, pado.rmat_edges(18, 4, seed=3))
    peak = []
    for pull_ratio in (0xFFFFFFFF, 0):
        ctx.trim()
        exp = _build(ctx, dg, wide, pull_ratio)
        peak.append(ctx.work_sizes()[1])
    single, four = peak
    # (blocks are at most a quarter larger than what they are taken for)
    room = single + single // 3
    print(f"[gpu] wide={wide}: batches of 1,024 take {single >> 20} MiB, of 4,096 {four >> 20} MiB", flush=True)
    assert room < four
    for limit in (room, (room + four) // 2, four - (1 << 20)):
        ctx.trim()
        ctx.set_work_limit(limit)
        got = _build(ctx, dg, wide)
        assert ctx.work_sizes()[0] == 0 and ctx.work_sizes()[1] <= limit
        assert all(np.array_equal(x, y) for x, y in zip(got, exp)), limit
        assert pado.lib().pado_gpu_last_error() == b""
    ctx.trim()
    ctx.set_work_limit(single // 2)
    with pytest.raises(pado.PadoError) as e:
        _build(ctx, dg, wide)
    assert e.value.status == 3
    ctx.set_work_limit(0)
    assert np.array_equal(_build(ctx, dg, wide)[3], exp[3])
    dg.close()
    ctx.close()


def test_label_pool_of_dense_label_sets():
    """A random graph with 4,100 labels a vertex, most lists long enough to grow
    by doubling.  A pool is made for twice the compacted lists (5/4 of the
    labels) and three times what a batch took (up to 5/2 of the labels), and the
    one before it is there while the lists move: 35 words a label at most.  By
    the steepest iteration, for as long as a batch could last, it was some 80."""
    rng = np.random.default_rng(1)
    n = 32000
    e = np.sort(rng.integers(0, n, (4_300_000, 2)), axis=1)
    e = np.unique(e[e[:, 0] != e[:, 1]], axis=0).astype(np.uint32)
    ctx = pado.Context(0)
    dg, _, _ = pado.DeviceGraph.from_edges(ctx, e)
    ctx.trim()
    got = _build(ctx, dg, False)
    peak, labels = ctx.work_sizes()[1], got[3].size
    fixed = 5 * 64 * 8 * n + 4096 * n  # rows of 64 words, root-distance table
    print(f"[gpu] {labels} labels, temporaries {peak >> 20} MiB", flush=True)
    assert peak <= 2 * fixed + 4 * 35 * labels
    ctx.trim()
    exp = _build(ctx, dg, False, 0xFFFFFFFF)
    assert all(np.array_equal(x, y) for x, y in zip(got, exp))
    dg.close()
    ctx.close()
