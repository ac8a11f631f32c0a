"""Child windows of a bounded match: the parent rows of a window are found on
the device, 64 probes a step.  Bounds around the window sizes (512 rows,
doubling), on joins whose levels hold from a few to several hundred thousand
rows, many of them without children: a bounded enumeration gives as many rows
as asked, all of them valid and distinct, and a bounded count min(count,
bound), at several lane counts, by both algorithms."""
import numpy as np
import pytest

import fsig_amd as F
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(130, 260), (2100, 5000), (33000, 90000)])
@pytest.mark.parametrize("lanes", [0, 4, 64])
def test_bounded_windows(gpu_ctx, n, m, lanes):
    g = F.HostGraph.chung_lu(n, m, 2.4, n).set_labels("uniform", 3, seed=7)
    off, adj, lab = g.arrays()
    q = F.Query(5, [0, 1, 2, 0, 1], [(0, 1), (1, 2), (2, 3), (3, 4)])
    dg = gpu_ctx.upload(g, pcsr=True)
    try:
        gpu_ctx.set_tune(lanes_per_row=lanes)
        total = F.match(dg, q, F.ALG_MMATCH, F.MODE_COUNT).count
        want, _ = O.match(q.labels, q.adjm(), off, adj, lab, threads=8, limit=1 << 30)
        assert total == want
        for alg in (F.ALG_MMATCH, F.ALG_GSI):
            for b in (1, 63, 511, 512, 513, 1025, 4096, 40001, 300007):
                print(n, lanes, alg, b, flush=True)
                assert F.match(dg, q, alg, F.MODE_COUNT, max_embeddings=b).count == min(want, b)
                r = F.match(dg, q, alg, F.MODE_ENUMERATE, max_embeddings=b, emb_cap=b)
                rows = r.embeddings
                assert r.count == len(rows) == min(want, b)
                if len(rows):
                    assert len(np.unique(rows, axis=0)) == len(rows)
                    assert all((lab[rows[:, c]] == q.labels[c]).all() for c in range(q.k))
                    for x, y in q.edges.tolist():  # every edge of every row is an adjacency entry
                        keys = np.repeat(np.arange(n, dtype=np.int64), np.diff(off.astype(np.int64))) * n + adj
                        assert np.isin(rows[:, x].astype(np.int64) * n + rows[:, y], keys).all()
                    assert all((rows[:, x] != rows[:, y]).all() for x in range(q.k) for y in range(x))
    finally:
        gpu_ctx.set_tune()
        dg.free()
