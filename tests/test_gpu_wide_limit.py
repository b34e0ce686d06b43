"""A wide index of 2^20 vertices, the most its labels' 20 hub bits hold: the
last-ranked vertex is hub 0xFFFFF, whose label words differ from the all-ones
padding of lists in the distance field alone.  A path of 8,001 vertices (4,000
hops on either side of its first-ranked vertex, so answers reach 8,000) and
isolated vertices; the last-ranked one is isolated, or the path's far end."""
import numpy as np
import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu

N, P = 1 << 20, 8001


def _bisection(p):
    """Positions of a path, the middle of each part before the part's halves."""
    order, parts = [], [(0, p)]
    for lo, hi in parts:
        if lo < hi:
            mid = (lo + hi) // 2
            order.append(mid)
            parts += [(lo, mid), (mid + 1, hi)]
    return np.array(order)


def _path(last_on_path):
    """(graph in rank space, id of each path position)."""
    ids = np.empty(P, np.int64)
    ids[_bisection(P)] = np.arange(P)
    if last_on_path:
        ids[P - 1] = N - 1
    a, b = np.concatenate([ids[:-1], ids[1:]]), np.concatenate([ids[1:], ids[:-1]])
    by = np.lexsort((-b, a))  # lists descending
    off = np.zeros(N + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(a, minlength=N))
    return pado.Graph(N, off, b[by].astype(np.uint32)), ids


@pytest.mark.parametrize("last_on_path", (False, True))
def test_last_vertex_of_a_full_wide_index(gpu_ctx, last_on_path):
    G, ids = _path(last_on_path)
    at = np.full(N, -1, np.int64)
    at[ids] = np.arange(P)
    dg = pado.DeviceGraph(gpu_ctx, G)
    W = pado.Index.build(gpu_ctx, dg, wide=True)
    W.order(np.arange(N, dtype=np.uint32))
    print(f"[gpu] last vertex on the path: {last_on_path}, {W.info.num_labels} labels", flush=True)
    last = np.uint32(N - 1)
    other = np.concatenate([ids, np.arange(P, P + 700), [N - 2, N - 1]]).astype(np.uint32)
    on = (at[last] >= 0) & (at[other] >= 0)
    exp = np.where(on, np.abs(at[other] - at[last]), np.where(other == last, 0, pado.WIDE_INF)).astype(np.uint16)
    if last_on_path:
        assert exp[on].max() == P - 1
    a = np.full(other.size, last, np.uint32)
    for rank_space in (True, False):
        for k in (other.size, 4096, 1000):  # groups of lanes, a wave per pair
            for s in range(0, other.size, k):
                x, y = a[s:s + k], other[s:s + k]
                assert np.array_equal(W.query(x, y, rank_space=rank_space), exp[s:s + k]), (rank_space, k, s)
                assert np.array_equal(W.query(y, x, rank_space=rank_space), exp[s:s + k]), (rank_space, k, s)
        for i in range(0, other.size, 997):
            assert W.query_pair(last, other[i], rank_space=rank_space) == exp[i], (rank_space, i)
    W.close()
    dg.close()
