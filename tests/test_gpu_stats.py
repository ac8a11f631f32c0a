"""Kernel statistics: what a match adds, a reset, a match from the static
scratch, and a thread that reads them while others match."""
import ctypes as C
import threading

import numpy as np
import pytest

import fsig_amd as F

pytestmark = pytest.mark.gpu

FAMILIES = range(len(F.KERNEL_FAMILIES))


def stats(ctx):
    return [{k: v for k, v in ctx.kernel_stats(f).items() if k != "ms"} for f in FAMILIES]


def graph():
    g = F.HostGraph.chung_lu(20000, 80000, 2.4, 3).set_labels("zipf", 4, 1.2, 4)
    dense = F.Query(4, [0, 1, 0, 2], [(0, 1), (1, 2), (0, 2), (2, 3)])
    path = F.Query(5, [0, 1, 0, 2, 0], [(i, i + 1) for i in range(4)])
    return g, [dense, path]


@pytest.mark.parametrize("alg", [F.ALG_MMATCH, F.ALG_GSI])
def test_each_match_adds_the_same_once(alg):
    g, qs = graph()
    ctx = F.Context(0, 1 << 30)
    dg = ctx.upload(g, pcsr=True)
    for q in qs:
        F.match(dg, q, alg)
        ctx.reset_stats()
        zero = stats(ctx)
        F.match(dg, q, alg)
        one = stats(ctx)
        again = stats(ctx)
        F.match(dg, q, alg)
        two = stats(ctx)
        off, adj = q.csr()
        sig = q.signature() if alg == F.ALG_GSI else None
        cnt = C.c_uint64(0)
        ctx.check(ctx._L.fsig_match_noalloc(ctx._h, dg._h, q.k, F._ptr(q.labels, F._i32p), F._ptr(off), F._ptr(adj),
                                            F._ptr(sig), alg, F.MODE_COUNT, 0, C.byref(cnt), F._ptr(None), 0))
        three = stats(ctx)
        ctx.reset_stats()
        assert all(v == 0 for s in zero + stats(ctx) for v in s.values())
        assert again == one
        joins = [one[F.KERNEL_FAMILIES.index(n)] for n in ("join_count", "join_tail")]
        assert any(s["alg_bytes"] and s["units"] for s in joins)
        assert two == [{k: 2 * v for k, v in s.items()} for s in one]
        assert three == [{k: 3 * v for k, v in s.items()} for s in one]
    dg.free()
    ctx.close()


def test_statistics_read_beside_matches():
    g, qs = graph()
    ctx = F.Context(0, 1 << 30)
    dg = ctx.upload(g)
    want = [F.match(dg, q).count for q in qs]
    stop, reads, errors = threading.Event(), [0], []

    def monitor():
        try:
            while not stop.is_set():
                ctx.kernel_stats(reads[0] % len(FAMILIES))
                reads[0] += 1
        except F.FsigError as e:
            errors.append(e)

    t = threading.Thread(target=monitor)
    t.start()
    try:
        got = [[F.match(dg, q).count for q in qs] for _ in range(60)]
        batch = [[int(c) for c in F.match_batch(dg, qs, bounds=[10 ** 10] * 2)[0]] for _ in range(20)]
    finally:
        stop.set()
        t.join()
    assert not errors and reads[0] > 0
    assert got == [want] * 60 and batch == [want] * 20
    dg.free()
    ctx.close()
