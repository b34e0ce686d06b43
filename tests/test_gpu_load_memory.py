"""Loading an index file takes the device memory of the index and a little
more: what most of it is, bit-parallel sets or weighted labels, is not held
twice."""
import ctypes
import threading

import numpy as np
import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def _free():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    # (the HIP runtime that the library itself uses)
    assert pado.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _load_and_watch(load):
    """What load() returns, the device memory it then holds and the most it held."""
    before = least = _free()
    done = threading.Event()

    def watch():
        nonlocal least
        while not done.is_set():
            least = min(least, _free())

    t = threading.Thread(target=watch)
    t.start()
    try:
        loaded = load()
    finally:
        done.set()
        t.join()
    return loaded, before - _free(), before - least


def test_load_holds_the_sets_once(gpu_ctx, tmp_path):
    edges = pado.rmat_edges(17, 4, seed=2)
    dg, rank, _ = pado.DeviceGraph.from_edges(gpu_ctx, edges)
    n = dg.num_v
    built = pado.Index.build(gpu_ctx, dg)
    built.order(rank)
    path = str(tmp_path / "index")
    built.store(path, rank)
    a, b = pado.uniform_pairs(n, 200000, seed=3)
    exp = built.query(a, b)
    pado.Index.load(gpu_ctx, path).close()  # (temporaries of this call stay for the next)
    gpu_ctx.sync()
    loaded, held, most = _load_and_watch(lambda: pado.Index.load(gpu_ctx, path))
    sets = n * 800
    print(f"[gpu] sets {sets >> 20} MiB, held {held >> 20}, at most {most >> 20}", flush=True)
    assert held >= sets
    assert most <= held + sets // 2
    assert np.array_equal(loaded.query(a, b), exp)
    loaded.close()
    built.close()
    dg.close()


def test_weighted_load_holds_the_labels_once(gpu_ctx, tmp_path):
    edges = pado.rmat_edges(15, 16, seed=2)
    w = pado.edge_weights(edges.shape[0], 1, 100, 9)
    dg, rank, _ = pado.DeviceGraph.from_edges(gpu_ctx, edges, w)
    n = dg.num_v
    built = pado.Index.build(gpu_ctx, dg)
    built.order(rank)
    path = str(tmp_path / "index").encode()
    L = pado.lib()
    L.pado_gpu_windex_store.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_char_p, ctypes.c_void_p, ctypes.c_uint32]
    L.pado_gpu_windex_load.argtypes = [ctypes.c_void_p, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p)]
    pado._check(L.pado_gpu_windex_store(gpu_ctx.h, built.h, path, pado._p(rank), n))
    a, b = pado.uniform_pairs(n, 200000, seed=3)
    exp = built.query(a, b)

    def load():
        h = ctypes.c_void_p()
        pado._check(L.pado_gpu_windex_load(gpu_ctx.h, path, ctypes.byref(h)))
        return pado.Index(gpu_ctx, h)

    load().close()
    gpu_ctx.sync()
    loaded, held, most = _load_and_watch(load)
    labels = loaded.info.num_labels
    print(f"[gpu] {labels} labels, held {held >> 20} MiB, at most {most >> 20}", flush=True)
    assert labels == built.info.num_labels and held >= 8 * labels
    assert most <= held + 4 * labels
    assert np.array_equal(loaded.query(a, b), exp)
    loaded.close()
    built.close()
    dg.close()
