"""Candidate-edge rows of degrees around the strides of every lane count and
around the hub limit, with all, some and none of their entries kept: stars
whose leaves alternate between two labels, beside a block that sets the
graph's mean degree (and with it the lanes of a row), with the class mask and,
from 2^20 vertices, with bitmaps.  Closed forms."""
import numpy as np
import pytest

import fsig_amd as F

pytestmark = pytest.mark.gpu

DEGREES = [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1030]


@pytest.mark.parametrize("n", [0, 1 << 20])
@pytest.mark.parametrize("block", [3, 400, 900])  # mean degrees 2, 20 and 91 (n = 0): 8, 16 and 64 lanes
def test_rows_of_all_lengths(gpu_ctx, block, n):
    hubs = DEGREES * 2  # leaves of the first half: labels 0 and 1 in turn; of the second: 0 only
    edges, label = [], [2] * len(hubs)
    for h, d in enumerate(hubs):
        for i in range(d):
            edges.append((h, len(label)))
            label.append(i % 2 if h < len(DEGREES) else 0)
    at = len(label)
    iu = np.stack(np.triu_indices(block, 1), 1) + at
    label += [3] * block
    label += [3] * max(0, n - len(label))
    g = F.HostGraph.from_edges(len(label), np.concatenate([np.asarray(edges), iu]).astype(np.uint32),
                               np.asarray(label, np.int32))
    dg = gpu_ctx.upload(g)
    zeros = [(d + 1) // 2 if h < len(DEGREES) else d for h, d in enumerate(hubs)]
    ones = [d - z for d, z in zip(hubs, zeros)]
    queries = {
        "edge 2-0": (F.Query(2, [2, 0], [(0, 1)]), sum(zeros)),
        "edge 2-1": (F.Query(2, [2, 1], [(0, 1)]), sum(ones)),
        "path 0-2-1": (F.Query(3, [0, 2, 1], [(0, 1), (1, 2)]), sum(z * o for z, o in zip(zeros, ones))),
        "path 0-2-0": (F.Query(3, [0, 2, 0], [(0, 1), (1, 2)]), sum(z * (z - 1) for z in zeros)),
        "triangle": (F.Query(3, [3, 3, 3], [(0, 1), (1, 2), (0, 2)]), block * (block - 1) * (block - 2)),
    }
    got = {}
    for nlf in (0, 1):
        gpu_ctx.set_tune(nlf_filter=nlf)
        for name, (q, _) in queries.items():
            got[name, nlf] = F.match(dg, q).count
            got[name, nlf, "batch"] = int(F.match_batch(dg, [q], bounds=[1 << 40])[0][0])
    gpu_ctx.set_tune()
    dg.free()
    assert got == {k: queries[k[0]][1] for k in got}


@pytest.mark.parametrize("n", [0, 1 << 20])
def test_unlabeled_rows(gpu_ctx, n):
    """Lists by degree of stars that share their leaves' ends: a centre keeps
    no leaf, a leaf keeps its centre; two leaves joined make a triangle."""
    edges, at = [], len(DEGREES)
    for h, d in enumerate(DEGREES):
        edges += [(h, at + i) for i in range(d)]
        edges += [(at + i, at + i + 1) for i in range(0, d - 1, 2)]
        at += d
    dg = gpu_ctx.upload(F.HostGraph.from_edges(max(at, n), np.asarray(edges, np.uint32)))
    got = [F.match(dg, F.Query(k, np.zeros(k, np.int32), e)).count
           for k, e in ((2, [(0, 1)]), (3, [(0, 1), (1, 2), (0, 2)]))]
    dg.free()
    assert got == [2 * len(edges), 6 * sum(d // 2 for d in DEGREES)]
