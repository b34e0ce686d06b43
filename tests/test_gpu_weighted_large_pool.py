"""A weighted build whose label pool goes past 2^31 words, so that offsets into
it need their 32nd bit: 300,000 vertices with 3 edges each, some 1.2 G labels."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.csgraph import dijkstra

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def test_pool_past_two_to_the_31():
    rng = np.random.default_rng(1)
    n = 300000
    edges = rng.integers(0, n, (450000, 2)).astype(np.uint32)
    w = pado.edge_weights(edges.shape[0], 1, 100, 3)
    ctx = pado.Context(0)
    dg, rank, _ = pado.DeviceGraph.from_edges(ctx, edges, w)
    n = dg.num_v
    idx = pado.Index.build(ctx, dg)
    held, grown, words = idx.holds()
    print(f"[gpu] {idx.info.num_labels} labels, pool of {words} words, held {held}, grown {grown}", flush=True)
    assert words > 1 << 31
    dg.close()
    idx.order(rank)
    e = np.sort(edges.astype(np.int64), axis=1)
    by = np.lexsort((w, e[:, 1], e[:, 0]))  # the lightest of parallel edges first
    e, ww = e[by], w[by].astype(float)
    first = np.ones(e.shape[0], bool)
    first[1:] = (e[1:] != e[:-1]).any(axis=1)
    A = sp.coo_matrix((ww[first], (e[first, 0], e[first, 1])), shape=(n, n)).tocsr()
    for s in rng.integers(0, n, 6):
        d = dijkstra(A, directed=False, indices=int(s))
        exp = np.where(np.isinf(d), float(pado.WINF), d).astype(np.uint32)
        assert np.array_equal(idx.query(np.full(n, s, np.uint32), np.arange(n, dtype=np.uint32)), exp), s
    idx.close()
    ctx.close()
