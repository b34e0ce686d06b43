"""Idle temporary memory: bounded over all contexts of a device, given back on
request, and a limit on what a context's calls have in use."""
import ctypes

import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def _memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    # (the HIP runtime that the library itself uses)
    assert pado.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value, total.value


def test_contexts_share_the_bound_and_trim_gives_back():
    # two builds that leave about 12 GB of temporaries each
    edges = pado.rmat_edges(20, 16, seed=1)
    ctxs = [pado.Context(0) for _ in range(2)]
    before, total = _memory()
    graphs = []
    for ctx in ctxs:
        dg, _, _ = pado.DeviceGraph.from_edges(ctx, edges)
        pado.Index.build(ctx, dg).close()
        graphs.append(dg)
    held = before - _memory()[0]
    own = 1 << 30  # the two graphs and the runtime's own allocations
    print(f"[gpu] held by two contexts: {held >> 20} MiB", flush=True)
    assert held <= total // 16 + own
    sizes = [ctx.work_sizes() for ctx in ctxs]
    print(f"[gpu] in use, peak, idle: {sizes}", flush=True)
    assert all(s[0] == 0 and s[1] > 4 << 30 for s in sizes)
    assert 0 < sum(s[2] for s in sizes) <= total // 16
    for ctx in ctxs:
        ctx.trim()
        assert ctx.work_sizes() == (0, 0, 0)
    assert before - _memory()[0] <= own
    # still usable, and its temporaries come back
    idx = pado.Index.build(ctxs[0], graphs[0])
    assert idx.info.num_labels > 0 and ctxs[0].work_sizes()[2] > 0
    idx.close()
    for dg, ctx in zip(graphs, ctxs):
        dg.close()
        ctx.close()


def test_limit_in_use():
    ctx = pado.Context(0)
    edges = pado.rmat_edges(12, 8, seed=1)
    ctx.set_work_limit(1 << 16)
    with pytest.raises(pado.PadoError) as e:
        pado.DeviceGraph.from_edges(ctx, edges)
    assert e.value.status == 3
    assert ctx.work_sizes()[0] == 0
    ctx.set_work_limit(0)
    dg, _, _ = pado.DeviceGraph.from_edges(ctx, edges)
    ctx.set_work_limit(1 << 20)
    with pytest.raises(pado.PadoError) as e:
        pado.Index.build(ctx, dg)
    assert e.value.status == 3
    ctx.set_work_limit(0)
    pado.Index.build(ctx, dg).close()
    ctx.close()
