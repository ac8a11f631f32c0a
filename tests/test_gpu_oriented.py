"""Counts of cliques, whose symmetry conditions go by degree and into the
candidate-edge lists: complete graphs (closed form n (n-1) .. (n-k+1)) with
shared intersections at the edges of the fused tail's tile and of its hash
set, power-law graphs and mixed patterns against the count of every embedding
(no symmetry conditions) and under a work limit (conditions by id)."""
import numpy as np
import pytest

import fsig_amd as F

pytestmark = pytest.mark.gpu


def clique(k, labels=None):
    e = [(a, b) for a in range(k) for b in range(a + 1, k)]
    return F.Query(k, np.zeros(k, np.int32) if labels is None else labels, e)


def count(dg, q, G=0, symmetry=0, limit=0, bound=0):
    dg.ctx.set_tune(lanes_per_row=G, symmetry=symmetry)
    dg.ctx.set_work_limit(limit)
    try:
        return F.match(dg, q, F.ALG_MMATCH, F.MODE_COUNT, max_embeddings=bound).count
    finally:
        dg.ctx.set_tune()
        dg.ctx.set_work_limit(0)


@pytest.mark.parametrize("k,n", [(3, n) for n in (3, 4, 33, 65, 342, 343, 684, 1026, 2049, 2051)] +
                         [(4, n) for n in (4, 5, 18, 66, 131, 260)])
def test_complete_graphs(gpu_ctx, k, n):
    iu = np.triu_indices(n, 1)
    dg = gpu_ctx.upload(F.HostGraph.from_edges(n, np.stack(iu, 1)))
    want = 1
    for i in range(k):
        want *= n - i
    got = {G: count(dg, clique(k), G) for G in ((0, 4, 16, 64) if n < 1000 else (0,))}
    got["bound"] = min(count(dg, clique(k), bound=want + 1), want)
    got["limit"] = count(dg, clique(k), limit=1 << 40)
    dg.free()
    assert all(v == want for v in got.values()), (want, got)


@pytest.mark.parametrize("k,scale,m", [(3, 13, 60000), (4, 12, 40000), (5, 10, 9000)])
def test_power_law(gpu_ctx, k, scale, m):
    dg = gpu_ctx.upload(F.HostGraph.rmat(scale, m, seed=3))
    want = count(dg, clique(k), symmetry=1)
    got = {G: count(dg, clique(k), G) for G in (0, 4, 8, 32, 64)}
    got["limit"] = count(dg, clique(k), limit=1 << 40)
    dg.free()
    assert want > 0 and all(v == want for v in got.values()), (want, got)


PATTERNS = {
    "prism": (6, [(0, 1), (1, 2), (0, 2), (3, 4), (4, 5), (3, 5), (0, 3), (1, 4), (2, 5)]),
    "bowtie": (5, [(0, 1), (1, 2), (0, 2), (2, 3), (3, 4), (2, 4)]),
    "triangle+tail": (4, [(0, 1), (1, 2), (0, 2), (2, 3)]),
    "clique4-pendant": (5, [(a, b) for a in range(4) for b in range(a + 1, 4)] + [(3, 4)]),
}


@pytest.mark.parametrize("name", sorted(PATTERNS))
def test_mixed_conditions(gpu_ctx, name):
    k, e = PATTERNS[name]
    g = F.HostGraph.rmat(9, 2200, seed=7)
    for labels in (np.zeros(k, np.int32), (np.arange(k) % 2).astype(np.int32)):
        dg = gpu_ctx.upload(g.set_labels("uniform", int(labels.max()) + 1, seed=5))
        q = F.Query(k, labels, e)
        want = count(dg, q, symmetry=1)
        got = {G: count(dg, q, G) for G in (0, 4, 16, 64)}
        got["limit"] = count(dg, q, limit=1 << 40)
        dg.free()
        assert all(v == want for v in got.values()), (name, want, got)
