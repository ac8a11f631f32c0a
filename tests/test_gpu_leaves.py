"""Leaves counted one lane per row: the product tail of alg 1 (the last two
vertices hang off earlier columns) and the per-candidate leaf counts of alg 2
(the last vertex hangs off one column).  Trees and pendant edges whose labels
repeat, so that leaves meet earlier vertices of their label in one class and
across classes, on graphs whose levels have fewer and more rows than either
rule asks for; bounded and unbounded, against the oracle and the level-by-
level count."""
import numpy as np
import pytest

import fsig_amd as F
import oracle as O

pytestmark = pytest.mark.gpu

QUERIES = {
    "star3": ([0, 1, 1, 1], [(0, 1), (0, 2), (0, 3)]),
    "star_two_labels": ([0, 1, 0, 1, 0], [(0, 1), (0, 2), (0, 3), (0, 4)]),
    "path5": ([0, 1, 0, 1, 0], [(0, 1), (1, 2), (2, 3), (3, 4)]),
    "path6": ([0, 0, 1, 1, 0, 0], [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5)]),
    "triangle_two_tails": ([0, 1, 0, 1, 1], [(0, 1), (1, 2), (0, 2), (0, 3), (2, 4)]),
    "cycle4_tails": ([0, 1, 0, 1, 0, 0], [(0, 1), (1, 2), (2, 3), (3, 0), (1, 4), (3, 5)]),
    "tail_of_tail": ([1, 0, 1, 0, 1], [(0, 1), (1, 2), (0, 2), (2, 3), (3, 4)]),
}
LIMIT = 30_000_000


@pytest.mark.parametrize("n,m", [(40, 90), (300, 900), (1500, 4500), (5000, 12000)])
@pytest.mark.parametrize("labels", [2, 3])
def test_leaf_counts(gpu_ctx, n, m, labels):
    g = F.HostGraph.chung_lu(n, m, 2.5, n + labels).set_labels("uniform", labels, seed=n + 1)
    off, adj, lab = g.arrays()
    dg = gpu_ctx.upload(g, pcsr=True)
    try:
        for name, (ql, e) in QUERIES.items():
            q = F.Query(len(ql), ql, e)
            want, _ = O.match(q.labels, q.adjm(), off, adj, lab, threads=8, limit=LIMIT)
            if want == O.TOO_MANY:
                continue
            print(n, labels, name, want, flush=True)
            for alg in (F.ALG_MMATCH, F.ALG_GSI):
                for fused in (0, 1):
                    for symmetry in (0, 1):
                        gpu_ctx.set_tune(fused_tail=fused, symmetry=symmetry)
                        got = F.match(dg, q, alg, F.MODE_COUNT).count
                        assert got == want, (name, alg, fused, symmetry)
                        bound = want // 2 + 1
                        got = F.match(dg, q, alg, F.MODE_COUNT, max_embeddings=bound).count
                        assert got == min(want, bound), (name, alg, fused, symmetry, "bounded")
    finally:
        gpu_ctx.set_tune()
        dg.free()
