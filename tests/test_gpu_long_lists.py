"""Fused tail over own lists around the length from which a whole group takes
them, read through or searched, beside short ones: triangles and 4-cycles of
complete multipartite graphs (closed forms), with the parts' ids in either
order, conditions by degree and (under a work limit) by id."""
import itertools

import numpy as np
import pytest

import fsig_amd as F

pytestmark = pytest.mark.gpu


def multipartite(parts):
    start = np.concatenate([[0], np.cumsum(parts)])
    e = []
    for i, j in itertools.combinations(range(len(parts)), 2):
        a, b = np.meshgrid(np.arange(start[i], start[i + 1]), np.arange(start[j], start[j + 1]))
        e.append(np.stack([a.ravel(), b.ravel()], 1))
    return F.HostGraph.from_edges(int(start[-1]), np.concatenate(e).astype(np.uint32))


def counts(dg, q, lanes=(0, 8, 16, 32, 64)):
    ctx, got = dg.ctx, {}
    for limit in (0, 1 << 60):
        for G in lanes:
            ctx.set_tune(lanes_per_row=G)
            ctx.set_work_limit(limit)
            got[limit != 0, G] = F.match(dg, q).count
    ctx.set_tune()
    ctx.set_work_limit(0)
    return got


@pytest.mark.parametrize("parts", [(1, 5, 511), (1, 5, 512), (1, 6, 506), (2, 40, 530), (1, 300, 700), (8, 8, 1100),
                                   (3, 513, 514), (70, 70, 1100)])
def test_triangles(gpu_ctx, parts):
    q = F.Query(3, np.zeros(3, np.int32), [(0, 1), (1, 2), (0, 2)])
    want = 6 * int(np.prod(parts))
    for order in (parts, parts[::-1], (parts[1], parts[2], parts[0])):
        dg = gpu_ctx.upload(multipartite(order))
        got = counts(dg, q)
        dg.free()
        assert all(v == want for v in got.values()), (order, want, got)


@pytest.mark.parametrize("a,b", [(3, 511), (3, 512), (3, 513), (65, 600), (20, 1100), (514, 515)])
def test_four_cycles(gpu_ctx, a, b):
    q = F.Query(4, np.zeros(4, np.int32), [(0, 1), (1, 2), (2, 3), (0, 3)])
    want = 2 * a * (a - 1) * b * (b - 1)
    for order in ((a, b), (b, a)):
        dg = gpu_ctx.upload(multipartite(order))
        got = counts(dg, q)
        dg.free()
        assert all(v == want for v in got.values()), (order, want, got)


@pytest.mark.parametrize("n,hub", [(4, 0), (24, 0), (25, 0), (26, 0), (25, 40), (26, 40), (3, 40), (120, 700)])
def test_longest_list_by_degree(gpu_ctx, n, hub):
    """K_n (its longest list by degree has n - 1 entries) beside a star whose
    centre's degree says nothing of its lists, on the edge of the rule for the
    tail's lanes; two triangles that share a vertex have a third list by id."""
    e = list(itertools.combinations(range(n), 2)) + [(n, n + 1 + i) for i in range(hub)]
    dg = gpu_ctx.upload(F.HostGraph.from_edges(n + 1 + hub, np.asarray(e, np.uint32)))
    tri = F.Query(3, np.zeros(3, np.int32), [(0, 1), (1, 2), (0, 2)])
    bowtie = F.Query(5, np.zeros(5, np.int32), [(0, 1), (1, 2), (0, 2), (2, 3), (3, 4), (2, 4)])
    got = [counts(dg, q) for q in (tri, bowtie)]
    dg.free()
    want = [n * (n - 1) * (n - 2), n * (n - 1) * (n - 2) * (n - 3) * (n - 4)]
    for g, w in zip(got, want):
        assert all(v == w for v in g.values()), (w, g)
