"""Weighted batches that the device holds for the host, and label pools that
are grown while a batch is held: that both happen is asserted, and the answers
equal Dijkstra's."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.csgraph import dijkstra

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def _chains():
    """A dense core, ranked first, and chains whose batches need more and more
    rounds than the batches before them."""
    rng = np.random.default_rng(5)
    parts, n = [np.stack(np.triu_indices(150, 1), 1)], 150
    for length in (3, 50, 5, 400, 1200):
        ids = np.concatenate([[rng.integers(0, 150)], np.arange(n, n + length)])
        parts.append(np.stack([ids[:-1], ids[1:]], 1))
        n += length
    return np.concatenate(parts).astype(np.uint32)


# R-MAT 16: 3.4 M labels in lists that grow by doubling; the first pool has 4.2 M words
@pytest.mark.parametrize("kind,grows", (("chains", False), ("labels", True)))
@pytest.mark.parametrize("batch", (0, 100))
def test_held_and_grown(gpu_ctx, kind, grows, batch):
    edges = _chains() if kind == "chains" else pado.rmat_edges(16, 16, seed=4).astype(np.uint32)
    w = pado.edge_weights(edges.shape[0], 1, 100, 9)
    dg, rank, _ = pado.DeviceGraph.from_edges(gpu_ctx, edges, w)
    n = dg.num_v
    idx = pado.Index.build(gpu_ctx, dg, batch_size=batch)
    held, grown, _ = idx.holds()
    print(f"[gpu] {kind} batch {batch}: {n} vertices, {idx.info.num_labels} labels, held {held}, grown {grown}",
          flush=True)
    assert held > 0 and (grown > 0) == grows
    idx.order(rank)
    e = np.sort(edges.astype(np.int64), axis=1)
    by = np.lexsort((w, e[:, 1], e[:, 0]))  # the lightest of parallel edges first
    e, ww = e[by], w[by].astype(float)
    first = np.ones(e.shape[0], bool)
    first[1:] = (e[1:] != e[:-1]).any(axis=1)
    A = sp.coo_matrix((ww[first], (e[first, 0], e[first, 1])), shape=(n, n)).tocsr()
    src = np.random.default_rng(1).integers(0, n, 12)
    d = dijkstra(A, directed=False, indices=src)
    exp = np.where(np.isinf(d), float(pado.WINF), d).astype(np.uint32).ravel()
    a, b = np.repeat(src, n).astype(np.uint32), np.tile(np.arange(n), src.size).astype(np.uint32)
    assert np.array_equal(idx.query(a, b), exp)
    idx.close()
    dg.close()
