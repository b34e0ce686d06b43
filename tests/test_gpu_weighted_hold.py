"""Weighted batches that are enqueued whole and then held: chains whose batches
need many more rounds than the ones before them, and label pools that fill up;
the answers against Dijkstra."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.csgraph import dijkstra

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def _graph(kind):
    rng = np.random.default_rng(4)
    if kind == "chains":  # a dense core first by degree, then chains of growing length
        core = np.stack(np.triu_indices(150, 1), 1)
        parts, n = [core], 150
        for length in (2, 3, 5, 9, 40, 2, 200, 700, 3, 1500):
            ids = np.concatenate([[rng.integers(0, 150)], np.arange(n, n + length)])
            parts.append(np.stack([ids[:-1], ids[1:]], 1))
            n += length
        return np.concatenate(parts).astype(np.uint32), n
    if kind == "grid":  # long searches in every batch
        return pado.grid_edges(60, 0.2, 3).astype(np.uint32), 3600
    edges = pado.rmat_edges(13, 40, seed=2).astype(np.uint32)  # many labels per vertex
    return edges, int(edges.max()) + 1


@pytest.mark.parametrize("kind", ("chains", "grid", "labels"))
@pytest.mark.parametrize("batch", (0, 512, 64, 7))
def test_held_batches(gpu_ctx, kind, batch):
    edges, n = _graph(kind)
    w = pado.edge_weights(edges.shape[0], 1, 100, 9)
    dg, rank, _ = pado.DeviceGraph.from_edges(gpu_ctx, edges, w)
    n = dg.num_v
    idx = pado.Index.build(gpu_ctx, dg, batch_size=batch)
    idx.order(rank)
    keep = {}
    for (x, y), ww in zip(edges.tolist(), w.tolist()):
        k = (min(x, y), max(x, y))
        keep[k] = min(ww, keep.get(k, 256))
    e = np.array(list(keep), np.int64)
    A = sp.coo_matrix((np.array(list(keep.values()), float), (e[:, 0], e[:, 1])), shape=(n, n)).tocsr()
    rng = np.random.default_rng(1)
    src = rng.integers(0, n, 40)
    d = dijkstra(A, directed=False, indices=src)
    exp = np.where(np.isinf(d), float(pado.WINF), d).astype(np.uint32).ravel()
    a, b = np.repeat(src, n).astype(np.uint32), np.tile(np.arange(n), 40).astype(np.uint32)
    print(f"[gpu] {kind} batch {batch}: {n} vertices, {idx.stats()['iterations']} rounds", flush=True)
    assert np.array_equal(idx.query(a, b), exp)
