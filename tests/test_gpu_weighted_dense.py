"""Weighted builds whose frontiers hold many roots per word: complete graphs and
stars around the sizes of words, edge chunks and batches, all pairs against
Dijkstra and the number of canonical labels."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.csgraph import dijkstra

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def _edges(kind, n):
    if kind == "complete":
        a, b = np.triu_indices(n, 1)
    else:  # a few hubs joined to everything
        a, b = (x.ravel() for x in np.meshgrid(np.arange(5), np.arange(5, n)))
    return np.stack([a, b], 1).astype(np.uint32)


@pytest.mark.parametrize("kind,n", [("complete", x) for x in (17, 33, 64, 65, 130, 515, 700)] +
                         [("hubs", x) for x in (21, 80, 300, 1200)])
def test_dense_frontiers(gpu_ctx, kind, n):
    edges = _edges(kind, n)
    w = pado.edge_weights(edges.shape[0], 1, 255, n)
    dg, rank, _ = pado.DeviceGraph.from_edges(gpu_ctx, edges, w)
    idx = pado.Index.build(gpu_ctx, dg)
    idx.order(rank)
    e = edges.astype(np.int64)
    A = sp.coo_matrix((w.astype(float), (e[:, 0], e[:, 1])), shape=(n, n)).tocsr()
    d = dijkstra(A, directed=False).astype(np.uint32)
    a, b = (x.ravel().astype(np.uint32) for x in np.meshgrid(np.arange(n), np.arange(n)))
    print(f"[gpu] {kind} {n}", flush=True)
    assert np.array_equal(idx.query(a, b), d[a, b])
    # canonical labels: r labels v iff no vertex ranked above r lies on a shortest v-r path
    by = np.empty((n, n), np.uint32)  # distances in rank space
    by[np.ix_(rank, rank)] = d
    want = 0
    for r in range(n):
        v = np.arange(r, n)
        via = (by[:r, v] + by[:r, [r]]).min(axis=0) if r else np.full(v.size, 0xFFFFFFFF, np.uint32)
        want += int((via > by[r, v]).sum())
    assert idx.stats()["num_labels"] == want
