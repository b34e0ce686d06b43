"""Bit-parallel sweep at the degrees where its work units change: vertices
that share a wave, fill one piece, or need several."""
import numpy as np
import pytest

import oracle
import parallel_distance_oracle_amd as pado
from helpers import rank_space

pytestmark = pytest.mark.gpu

DEGREES = (1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 300)


def _edges(seed):
    """For each degree a few centres with exactly that many neighbours; leaves
    are shared and joined at random, so siblings and several parents occur."""
    rng = np.random.default_rng(seed)
    centres = [d for d in DEGREES for _ in range(6)]
    first_leaf = len(centres)
    leaves = 700
    edges = set()
    for c, d in enumerate(centres):
        for v in rng.choice(leaves, d, replace=False):
            edges.add((c, first_leaf + int(v)))
    for a, b in rng.integers(0, leaves, (900, 2)):
        if a != b:
            edges.add((first_leaf + int(min(a, b)), first_leaf + int(max(a, b))))
    # two more components, and a path for depth
    n = first_leaf + leaves
    edges |= {(n + i, n + i + 1) for i in range(60)}
    edges |= {(n + 61, n + 62 + i) for i in range(17)}
    return np.array(sorted(edges), np.uint32)


@pytest.mark.parametrize("seed", (1, 2))
@pytest.mark.parametrize("wide", (False, True))
def test_records_equal_oracle(gpu_ctx, seed, wide):
    G, rank, _ = rank_space(_edges(seed))
    dg = pado.DeviceGraph(gpu_ctx, G)
    print(f"[gpu] n={G.num_v} wide={wide}", flush=True)
    got = pado.Index.build(gpu_ctx, dg, wide=wide).export()
    exp = oracle.Index(G.num_v, G.off, G.adj)
    assert np.array_equal(got[0], exp.bp_d) and np.array_equal(got[1], exp.bp_s)
    assert np.array_equal(got[2], exp.loff) and np.array_equal(got[3], exp.hub)
    assert np.array_equal(got[4].astype(np.int64), np.asarray(exp.dist).astype(np.int64))
