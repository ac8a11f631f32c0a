"""Digests folded in as the last level is found: every lane count, both
algorithms, queries of 1..9 vertices whose last join vertex has no, one or
several backward neighbours, wherever it stands in query order.  Exact
equality with the oracle's digest."""
import numpy as np
import pytest

import fsig_amd as F
import oracle as O
from fsig_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [0, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("n,labels", [(700, 3), (3001, 9)])
def test_digest_of_the_last_level(gpu_ctx, lanes, n, labels):
    g = F.HostGraph.chung_lu(n, 4 * n, 2.4, 31 + n).set_labels("uniform", labels, seed=32)
    off, adj, lab = g.arrays()
    qs = [q for _, q in W.walk_queries(g, 8, 3, 6, 33)] + [q for _, q in W.walk_queries(g, 2, 8, 9, 34)]
    qs = [q for q in qs if q.k >= 4 or n > 1000]
    qs.append(F.Query(1, [1], np.zeros((0, 2))))
    qs.append(F.Query(2, [0, 1], [(0, 1)]))
    qs.append(F.Query(3, [0, 1, 2], [(0, 1)]))                    # last vertex without a neighbour
    qs.append(F.Query(4, [1, 0, 0, 1], [(0, 3), (1, 2), (2, 3), (0, 1)]))
    dg = gpu_ctx.upload(g, pcsr=True)
    done = 0
    try:
        gpu_ctx.set_tune(lanes_per_row=lanes)
        for q in qs:
            if F.match(dg, q, F.ALG_MMATCH, F.MODE_COUNT, max_embeddings=3_000_001).count > 3_000_000:
                continue
            want = O.match_digest(q.labels, q.adjm(), off, adj, lab, threads=8)
            for alg in (F.ALG_MMATCH, F.ALG_GSI):
                print(n, lanes, q.k, q.num_edges, alg, flush=True)
                assert F.match_digest(dg, q, alg) == want, (q.labels.tolist(), q.edges.tolist(), alg)
            done += 1
    finally:
        gpu_ctx.set_tune()
        dg.free()
    assert done >= 8
