"""Work that users of the engine have it do, as timed cases.

Two families of cases:

  given query     a data graph generated from the seed, uploaded, and one
                  query: the diamond of a seeded walk, one of the two 8-vertex
                  queries of the dblp-shaped workload, or an unlabeled
                  pattern.  Counted (alg 1 or alg 2), enumerated to host rows,
                  or enumerated into the set digest.
  resident graph  one data graph per shape stays resident, as in a service;
                  the seed draws the random-walk queries that are asked of it,
                  each with a bound ("more than L?") and under a work limit:
                  one `match` after another, one bounded batch, or a served
                  stream.

Graph laws, query laws, bounds and the work limit are those of
fsig_amd/workloads.py.  Counts, candidate-set sizes, rows, digests and
statuses are whole numbers.
"""
import math

import numpy as np

import fsig_amd as F
from fsig_amd import workloads as W

WORK_LIMIT = W.C4_QUERIES["work_limit"]
BOUND = W.C4_QUERIES["bound"]

# The 8-vertex walk queries of the dblp-shaped workload (workloads.c2_queries):
# 12 edges, and a path.  Given here so that graphs of other seeds are asked
# the same query.
DBLP_QUERIES = {
    "dense": ([0, 6, 3, 0, 9, 1, 1, 0], [(0, 1), (1, 2), (1, 3), (1, 5), (1, 6), (2, 3), (3, 4), (3, 5), (3, 6),
                                        (4, 5), (5, 6), (6, 7)]),
    "sparse": ([1, 5, 2, 12, 0, 1, 7, 2], [(i, i + 1) for i in range(7)]),
}


def listed():
    return [
        # Smallest calls: a 4-vertex query on a 10,000-vertex graph (a lookup
        # in an interactive program).  Launches, synchronisations and latency
        # count; rows to the host with alg 1, a count with alg 2.
        dict(name="diamond_rows", kind="diamond", n=10000, m=50000, labels=8, alg=1, mode="rows"),
        dict(name="diamond_gsi", kind="diamond", n=10000, m=50000, labels=8, alg=2, mode="count"),
        # Exact counts of one labeled query on a dblp-sized graph: the usual
        # use of the matcher, dense (intersections) and sparse (a path: many
        # partial embeddings), with each of the two algorithms.
        dict(name="dblp_dense", kind="dblp", query="dense", n=317080, m=1049866, labels=16, alg=1, mode="count"),
        dict(name="dblp_sparse", kind="dblp", query="sparse", n=317080, m=1049866, labels=16, alg=1, mode="count"),
        dict(name="dblp_dense_gsi", kind="dblp", query="dense", n=317080, m=1049866, labels=16, alg=2, mode="count"),
        # Enumeration instead of a count: every embedding is materialised on
        # the device and folded into the set digest.
        dict(name="dblp_digest", kind="dblp", query="dense", n=200001, m=600000, labels=16, alg=1, mode="digest"),
        # Motif counts on unlabeled power-law graphs: no label filter, hubs,
        # long lists.  The triangle is set up and one intersection per edge,
        # the 4-clique a deeper join with symmetry conditions.
        dict(name="rmat_triangle", kind="pattern", pattern="triangle", scale=20, m=8750000, mode="count"),
        dict(name="rmat_clique4", kind="pattern", pattern="clique4", scale=18, m=2187500, mode="count"),
        # 16 walk queries of 4..16 vertices on a 1M-vertex graph, one call each.
        dict(name="cl1m_loop", kind="walks", law="chung_lu", n=1000000, m=10000000, labels=32, kmin=4, kmax=16,
             queries=16, how="loop"),
        # 48 of them in one bounded batch.
        dict(name="cl1m_batch", kind="walks", law="chung_lu", n=1000000, m=10000000, labels=32, kmin=4, kmax=16,
             queries=48, how="batch"),
        # The largest graph: 16.8M vertices, 200M edges, queries of up to 32
        # vertices, one call each, and as a served stream.
        dict(name="rmat16m_loop", kind="walks", law="rmat", scale=24, m=200000000, labels=64, kmin=4, kmax=32,
             queries=8, how="loop"),
        dict(name="rmat16m_served", kind="walks", law="rmat", scale=24, m=200000000, labels=64, kmin=4, kmax=32,
             queries=32, how="served"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["diamond", "dblp", "pattern", "walks", "walks"])
    if kind == "diamond":
        n = _log(rng, 2000, 200000)
        alg, mode = rng.choice([(1, "rows"), (1, "count"), (1, "digest"), (2, "rows"), (2, "count")])
        return dict(kind=kind, n=n, m=int(n * rng.uniform(4, 6)), labels=rng.randint(3, 17), alg=alg, mode=mode)
    if kind == "dblp":
        n = _log(rng, 30000, 317080)
        query = rng.choice(["dense", "sparse"])
        alg, mode = rng.choice([(1, "count"), (1, "count"), (2, "count"), (1, "digest")])
        if mode == "digest" or alg == 2:
            n = min(n, 60000 + n // 4)
        return dict(kind=kind, query=query, n=n, m=int(n * rng.uniform(2.8, 3.3)), labels=16, alg=alg, mode=mode)
    if kind == "pattern":
        pattern, top = rng.choice([("triangle", 20), ("clique4", 18), ("cycle4", 16), ("house", 12)])
        scale = rng.randint(max(10, top - 4), top)
        return dict(kind=kind, pattern=pattern, scale=scale, m=int((1 << scale) * rng.uniform(5, 8.3)), mode="count")
    how = rng.choice(["loop", "batch", "served"])
    c = dict(kind="walks", how=how, labels=rng.choice([16, 32, 33, 64, 100]), kmin=4, kmax=rng.randint(6, 32),
             queries=rng.randint(4, 16))
    if rng.random() < 0.5:
        n = _log(rng, 30000, 1000000)
        c.update(law="chung_lu", n=n, m=int(n * rng.uniform(3, 10)))
    else:
        scale = rng.randint(15, 20)
        c.update(law="rmat", scale=scale, m=int((1 << scale) * rng.uniform(5, 12)))
    return c


# ---------------------------------------------------------------------------
# What a program keeps: one context, and for a resident graph the graph and
# (served) the server over it.  One resident graph at a time.
_ctx = None
_resident = {}


def _context():
    global _ctx
    if _ctx is None:
        _ctx = F.Context(0, 32 << 30)
    return _ctx


def _shape(case):
    return tuple(sorted((k, v) for k, v in case.items() if k in ("law", "n", "scale", "m", "labels")))


def _resident_graph(case):
    key = _shape(case)
    if _resident.get("key") != key:
        if "server" in _resident:
            _resident["server"].close()
        _resident.clear()
        if case["law"] == "chung_lu":
            g = F.HostGraph.chung_lu(case["n"], case["m"], 2.3, 5).set_labels("zipf", case["labels"], 1.2, 6)
        else:
            g = F.HostGraph.rmat(case["scale"], case["m"], 0.57, 0.19, 0.19, 8).set_labels(
                "uniform", case["labels"], seed=9)
        _resident.update(key=key, dg=_context().upload(g))
    return _resident["dg"]


def _server(dg):
    if "server" not in _resident:
        _resident["server"] = F.Server(dg, workers=6, hbm_budget=96 << 30, max_batch=32)
        _resident["server"].set_work_limit(WORK_LIMIT)
    return _resident["server"]


def _given(case, seed):
    """Host graph and query of a given-query case."""
    if case["kind"] == "pattern":
        g = F.HostGraph.rmat(case["scale"], case["m"], 0.57, 0.19, 0.19, seed)
        k, e = W.C3_PATTERNS[case["pattern"]]
        return g, F.Query(k, np.zeros(k, np.int32), e)
    if case["kind"] == "diamond":
        g = F.HostGraph.chung_lu(case["n"], case["m"], 2.5, seed).set_labels("uniform", case["labels"], seed=seed + 1)
        try:
            return g, g.walk_query(4, 5, 5, seed=seed + 2)
        except F.FsigError:  # no walk closes a diamond on this graph: any four vertices a walk meets
            return g, g.walk_query(4, 3, 6, seed=seed + 2)
    g = F.HostGraph.chung_lu(case["n"], case["m"], 2.3, seed).set_labels("zipf", case["labels"], 1.2, seed + 1)
    labels, edges = DBLP_QUERIES[case["query"]]
    return g, F.Query(8, labels, edges)


ROWS_CAP = 1 << 17


def prepare(case, seed):
    ctx = _context()
    if case["kind"] != "walks":
        g, q = _given(case, seed)
        rows = np.zeros((ROWS_CAP, q.k), np.uint32) if case["mode"] == "rows" else None
        return dict(case=case, dg=ctx.upload(g, pcsr=case.get("alg", 1) == 2), queries=[q], rows=rows)
    dg = _resident_graph(case)
    qs = [q for _, q in W.walk_queries(dg.host, case["queries"], case["kmin"], case["kmax"], seed, log_uniform=True,
                                       max_attempts=200, alternate_drawn=True)]
    # each caller asks "more than L?" with an L of its own
    bounds = np.exp(np.random.default_rng(seed).uniform(math.log(BOUND / 100), math.log(BOUND), len(qs)))
    state = dict(case=case, dg=dg, queries=qs, bounds=[int(b) for b in bounds])
    if case["how"] == "served":
        state["server"] = _server(dg)
    return state


def run(state):
    case, dg, qs = state["case"], state["dg"], state["queries"]
    if case["kind"] != "walks":
        q, alg = qs[0], case.get("alg", 1)
        if case["mode"] == "digest":
            count, digest = F.match_digest(dg, q, alg)
            return dict(count=count, digest=[d - (1 << 64) if d >> 63 else d for d in digest])
        if case["mode"] == "rows":
            r = F.match(dg, q, alg, F.MODE_ENUMERATE, emb_cap=ROWS_CAP)
            state["rows"][:len(r.embeddings)] = r.embeddings  # the program's own table
            return dict(count=r.count, candidates=r.candidates, rows=state["rows"])
        r = F.match(dg, q, alg, F.MODE_COUNT)
        return dict(count=r.count, candidates=r.candidates)
    bounds = state["bounds"]
    if case["how"] == "loop":
        dg.ctx.set_work_limit(WORK_LIMIT)
        counts, cand = np.zeros(len(qs), np.int64), np.zeros((len(qs), case["kmax"]), np.uint32)
        for i, (q, b) in enumerate(zip(qs, bounds)):
            try:
                r = F.match(dg, q, F.ALG_MMATCH, F.MODE_COUNT, max_embeddings=b)
                counts[i] = r.count
                cand[i, :q.k] = r.candidates
            except F.FsigError as e:  # refused: the search is over the work limit
                if e.code != F.FSIG_ELIMIT:
                    raise
                counts[i] = -1
        dg.ctx.set_work_limit(0)
        return dict(counts=counts, candidates=cand)
    if case["how"] == "batch":
        dg.ctx.set_work_limit(WORK_LIMIT)
        counts, _, status = F.match_batch(dg, qs, bounds=bounds, status=True)
        dg.ctx.set_work_limit(0)
        return dict(counts=counts.astype(np.int64), status=status)
    server = state["server"]
    tickets = [server.submit(q, b) for q, b in zip(qs, bounds)]
    counts = []
    for t in tickets:
        try:
            counts.append(server.wait(t)[0])
        except F.FsigError as e:
            if e.code != F.FSIG_ELIMIT:
                raise
            counts.append(-1)
    return dict(counts=np.array(counts, np.int64))


def work(case):
    """The graph read once (offsets, labels, adjacency) per query; a digest
    also reads no less.  Operations: one membership test per adjacency entry."""
    n = case["n"] if "n" in case else 1 << case["scale"]
    reads = 8 * n + 8 * case["m"]
    q = case.get("queries", 1)
    return dict(bytes=float(reads) * q, flops=2.0 * case["m"] * q)


# ---------------------------------------------------------------------------
def _numpy_join(g, q, most=20_000_000):
    """Number of embeddings by level-wise expansion in numpy, or None when a
    level passes `most` rows."""
    off, adj, lab = (a.astype(np.int64) for a in g.arrays())
    keys = np.repeat(np.arange(g.n, dtype=np.int64), np.diff(off)) * g.n + adj  # ascending
    nbrs = {v: set() for v in range(q.k)}
    for a, b in q.edges.tolist():
        nbrs[a].add(b)
        nbrs[b].add(a)
    order = [0]
    while len(order) < q.k:
        order.append(max((v for v in range(q.k) if v not in order), key=lambda v: len(nbrs[v] & set(order))))
    rows = np.nonzero(lab == q.labels[order[0]])[0].reshape(-1, 1)
    for p in range(1, q.k):
        w = order[p]
        back = [c for c in range(p) if order[c] in nbrs[w]]
        if not back or not len(rows):
            return None if len(rows) else 0
        src = rows[:, back[0]]
        deg = off[src + 1] - off[src]
        if int(deg.sum()) > most:
            return None
        rep = np.repeat(np.arange(len(rows)), deg)
        x = adj[np.repeat(off[src] - np.concatenate([[0], np.cumsum(deg)[:-1]]), deg) + np.arange(int(deg.sum()))]
        ok = lab[x] == q.labels[w]
        rep, x = rep[ok], x[ok]
        for c in back[1:]:
            key = rows[rep, c] * g.n + x
            at = np.minimum(np.searchsorted(keys, key), len(keys) - 1)
            ok = keys[at] == key
            rep, x = rep[ok], x[ok]
        for c in range(p):
            ok = rows[rep, c] != x
            rep, x = rep[ok], x[ok]
        rows = np.concatenate([rows[rep], x[:, None]], axis=1)
    return len(rows)


def exact(case, seed):
    """The count where a plain join is small enough; other outputs (candidate
    sizes, rows in the engine's order, digests) are its own."""
    if case["kind"] != "diamond":
        return None
    count = _numpy_join(*_given(case, seed))
    if case["mode"] == "digest":
        return dict(count=count, digest=[None, None])
    return dict(count=count, candidates=None, **({"rows": None} if case["mode"] == "rows" else {}))
