"""The relaxations of a weighted build, counted: with equal weights every
(vertex, root) pair improves once, at its hop distance, so the build relaxes
exactly the edges of the pairs that earlier batches do not prune."""
import numpy as np
import pytest

import parallel_distance_oracle_amd as pado

pytestmark = pytest.mark.gpu


def _expected(n, off, adj, starts, loff, hub, dist):
    """Edges to vertices ranked below the root, over all pairs that a root's
    search reaches through pairs that hubs before its batch do not prune."""
    lists = [dict(zip(hub[int(loff[v]):int(loff[v + 1])].tolist(), dist[int(loff[v]):int(loff[v + 1])].tolist()))
             for v in range(n)]
    nbr = [adj[int(off[v]):int(off[v + 1])] for v in range(n)]
    total = 0
    for r in range(n):
        rs = max(s for s in starts if s <= r)
        mine = {h: d for h, d in lists[r].items() if h < rs}
        seen, front, d = {r}, [r], 0
        while front:
            nxt, d = [], d + 1
            for v in front:
                for t in nbr[v].tolist():
                    if t <= r:
                        continue
                    total += 1
                    if t in seen:
                        continue
                    seen.add(t)
                    if any(h in mine and mine[h] + x <= d for h, x in lists[t].items()):
                        continue
                    nxt.append(t)
            front = nxt
    return total


@pytest.mark.parametrize("n,deg,seed", ((200, 6, 1), (700, 5, 2), (900, 24, 3)))
def test_relaxations(gpu_ctx, n, deg, seed):
    rng = np.random.default_rng(seed)
    e = np.sort(rng.integers(0, n, (n * deg // 2, 2)), axis=1)
    e = np.unique(e[e[:, 0] != e[:, 1]], axis=0).astype(np.uint32)
    dg, _, _ = pado.DeviceGraph.from_edges(gpu_ctx, e, np.ones(e.shape[0], np.uint32))
    n = dg.num_v
    off, adj, _ = dg.export()
    idx = pado.Index.build(gpu_ctx, dg)
    loff, hub, dist = idx.wexport()
    starts = [0] + list(range(64, n, 512))  # the first batch has an eighth of the roots
    exp = _expected(n, off, adj, starts, loff, hub, dist)
    print(f"[gpu] {n} vertices: {idx.stats()['pushes']} relaxations, expected {exp}", flush=True)
    assert idx.stats()["pushes"] == exp
    idx.close()
    dg.close()
