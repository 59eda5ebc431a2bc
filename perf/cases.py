"""The work that users of beep_amd have it do, as cases that can be timed.

A case is a data graph (a deterministic generator with its sizes), one or more
queries ("pattern:task") and the entry point they go through:

  count    Prepared.count: counting on a graph that is resident in HBM
  hash     the same with every match walked and hashed (sgm match sets)
  buffer   the same with the first match_cap tuples returned
  batch    Batch.run: all queries as one captured graph
  serve    Server.submit / poll: all queries submitted at once, then collected
  oneshot  SG_Match.run: preparation, upload and counting of a graph in host
           memory, what the command line and a reference-style driver do

Graphs are R-MAT (.57, .19, .19, .05) and Chung-Lu, as in beep_amd.workloads,
the benchmark and the tests.
"""
import math

import numpy as np
import torch

import beep_amd as B
from beep_amd import patterns as P

RMAT = (0.57, 0.19, 0.19)


def _rmat(scale, samples, **more):
    return dict(kind="rmat", scale=scale, samples=samples, **more)


def _chung_lu(n, samples, gamma=2.2, i0=3.5, **more):
    return dict(kind="chung_lu", n=n, samples=samples, gamma=gamma, i0=i0, **more)


def listed():
    return [
        # The smallest call: a graph of a few thousand edges, as an interactive
        # user or a loop over many small graphs counts them; launches and waits.
        dict(_rmat(10, 8 << 10), name="rmat10_triangle", queries="triangle:sgc", entry="count"),
        # The triangle count of the small R-MAT workload (rmat16).
        dict(_rmat(16, 16 << 16), name="rmat16_triangle", queries="triangle:sgc", entry="count"),
        # Returning a match set: every triangle of a 20,000-vertex graph into
        # the caller's buffer.
        dict(_chung_lu(20000, 60000, i0=5.0), name="chunglu20k_buffer", queries="triangle:sgm", entry="buffer",
             match_cap=1 << 17),
        # Verifying a match set: a five-vertex pattern whose matches are all
        # walked and hashed; hubs with donated subtrees.
        dict(_chung_lu(20001, 60000, i0=5.0), name="chunglu20k_w5_hash", queries="w5:sgm", entry="hash"),
        # The benchmark's two queries on its com-youtube-sized graph.
        dict(_chung_lu(1134890, 3070000), name="chunglu1m_4clique", queries="4clique:sgm", entry="count"),
        dict(_chung_lu(1134890, 3070000), name="chunglu1m_diamond", queries="diamond:sgm", entry="count"),
        # Match sets at the benchmark's size: 4-cliques walked and hashed.
        dict(_chung_lu(1134890, 3070000), name="chunglu1m_4clique_hash", queries="4clique:sgm", entry="hash"),
        # Deeper patterns on skewed graphs: cliques (every level intersects) on
        # the whole rmat22cut workload, the largest graph here ...
        dict(_rmat(22, 17_030_000, n_keep=3774768), name="rmat22cut_5clique", queries="5clique:sgc", entry="count"),
        # ... and the hub + 4-cycle wheel (hubs, paired last levels) on a
        # quarter of it.
        dict(_rmat(20, 17 << 18), name="rmat20_w5", queries="w5:sgc", entry="count"),
        # The eight named patterns of the batched workload as one captured graph.
        dict(_rmat(17, 17 << 15), name="rmat17_batch8",
             queries="triangle:sgc,tailed_triangle:sgc,diamond:sgc,4clique:sgc,4star:sgc,w5:sgc,5clique:sgc,6clique:sgc",
             entry="batch"),
        # The serving loop: a burst of small patterns over one resident graph of
        # the serving workload's density (a tenth of chunglu3m), one in five
        # returning a match-set hash.
        dict(_chung_lu(30724, 1213500, gamma=2.0, i0=70.0), name="chunglu30k_serve",
             queries="triangle:sgc,wedge:sgm,4star:sgc,tailed_triangle:sgm,diamond:sgc,4clique:sgm,"
                     "triangle:sgm:hash,diamond:sgm,tailed_triangle:sgc,4clique:sgc",
             entry="serve"),
        # From a graph in host memory to a count, once: what the command line does.
        dict(_chung_lu(200000, 540000), name="chunglu200k_oneshot", queries="diamond:sgm", entry="oneshot"),
    ]


def draw(rng):
    """One more case of the ranges above: graph sizes over their logarithm
    (2^9 to 2^20 vertices), every pattern and entry point, odd sizes."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    entry = rng.choice(["count", "count", "count", "count", "hash", "buffer", "batch", "serve", "oneshot"])
    small = ["triangle", "wedge", "tailed_triangle", "diamond", "4clique", "4star"]
    task = rng.choice(["sgm", "sgc"])
    more = {}
    if entry == "count":
        pattern = rng.choice(small + ["diamond", "4clique", "5clique", "w5"])
        top = 1 << 18 if pattern == "w5" else 1 << 20
        queries = f"{pattern}:{task}"
    elif entry in ("hash", "buffer"):
        queries, top = rng.choice(["triangle", "4clique"]) + ":sgm", 1 << 17
        if entry == "buffer":  # a buffer that holds every match
            queries, top, more["match_cap"] = "triangle:sgm", 1 << 14, 1 << 20
    else:
        names = rng.sample(small, 1 if entry == "oneshot" else rng.randint(2, 5))
        queries, top = ",".join(f"{q}:{rng.choice(['sgm', 'sgc'])}" for q in names), 1 << 17
    n = log_int(1 << 9, top)
    per = rng.uniform(2.5, 6.0)  # samples per vertex
    if rng.random() < 0.5:
        g = _rmat(max(9, min(20, round(math.log2(n)))), int(n * per), **more)
    else:
        g = _chung_lu(n | 1, int(n * per), gamma=round(rng.uniform(2.1, 2.6), 2), i0=round(rng.uniform(3.0, 8.0), 1), **more)
    return dict(g, queries=queries, entry=entry)


def _graph(case, seed):
    if case["kind"] == "rmat":
        return B.Graph.rmat(case["scale"], case["samples"], *RMAT, seed, case.get("n_keep", 0))
    return B.Graph.chung_lu(case["n"], case["samples"], case["gamma"], case["i0"], seed)


def _queries(case):
    """[(pattern, task, emit hash?), ...]"""
    return [tuple((q.split(":") + [""])[:3]) for q in case["queries"].split(",")]


def _plan(pattern, task):
    return B.Plan.from_edges(*P.directed(P.read_mtx_edges(pattern)), B.mode_of(task))


def prepare(case, seed):
    g = _graph(case, seed)
    plans = [_plan(q, task) for q, task, _ in _queries(case)]
    state = dict(case=case, plans=plans)
    entry = case["entry"]
    if entry == "oneshot":
        state.update(graph=g, matcher=B.SG_Match(_queries(case)[0][1]))
    elif entry == "serve":
        s = B.Server(g, lanes=4, pool_bytes=4 << 30)
        for p in plans:
            s.prepare(p)
        state.update(server=s, emits=[B.EMIT_HASH if h else B.EMIT_NONE for _, _, h in _queries(case)])
    else:
        preps = [B.Prepared(g, p) for p in plans]
        for pp in preps:
            pp.upload(0)
        state.update(preps=preps)
        if entry == "batch":
            state.update(batch=B.Batch(preps))
    return state


def _whole(*values):
    return np.array(values, dtype=np.uint64)


def run(state):
    case = state["case"]
    entry = case["entry"]
    if entry == "oneshot":
        return {"count": _whole(state["matcher"].run(state["graph"], state["plans"][0]))}
    if entry == "serve":
        server = state["server"]
        at = {server.submit(p, emit=e): i for i, (p, e) in enumerate(zip(state["plans"], state["emits"]))}
        done = [None] * len(at)
        for _ in at:
            r = server.poll()
            done[at[r["ticket"]]] = r
        return {"count": _whole(*[r["count"] for r in done]), "hash": _whole(*[r["hash_sum"] for r in done])}
    if entry == "batch":
        res, _ = state["batch"].run()
        return {"count": _whole(*[r["count"] for r in res])}
    pp = state["preps"][0]
    if entry == "count":
        return {"count": _whole(pp.count()["count"])}
    if entry == "hash":
        r = pp.count(emit=B.EMIT_HASH)
        return {"count": _whole(r["count"]), "hash": _whole(r["hash_sum"], r["hash_xor"])}
    r = pp.count(emit=B.EMIT_BUFFER, match_cap=case["match_cap"])
    # tuples come in no fixed order: as a set, i.e. by their packed ids
    m = r["matches"].astype(np.uint64)
    key = m[:, 0]
    for c in range(1, m.shape[1]):
        key = key << np.uint64(64 // m.shape[1]) | m[:, c]
    whole = np.zeros(case["match_cap"], dtype=np.uint64)
    whole[:len(key)] = np.sort(key)
    return {"count": _whole(r["count"]), "hash": _whole(r["hash_sum"], r["hash_xor"]), "matches": whole}


def work(case):
    """Each row entry and row pointer of the graph read once by every query; a
    pass from host memory also writes the oriented rows to the card once."""
    n = case.get("n") or 1 << case["scale"]
    graph = 8 * case["samples"] + 8 * n
    reads = len(_queries(case)) * (2 if case["entry"] == "oneshot" else 1)
    return {"bytes": graph * reads, "flops": 0}


# ---------------------------------------------------------------------------
# What the counts have to be, from the generators' definition and plain tensor
# arithmetic on edge lists.


def _uniforms(seed, samples, count):
    """`count` doubles in [0, 1) per sample: xoshiro256** seeded by splitmix64."""
    with np.errstate(over="ignore"):
        c = np.uint64
        x = c(seed & (1 << 64) - 1) * c(0xD1342543DE82EF95) + np.arange(samples, dtype=np.uint64) * c(0x9E3779B97F4A7C15) + c(1)
        s = []
        for _ in range(4):
            x = x + c(0x9E3779B97F4A7C15)
            z = (x ^ x >> c(30)) * c(0xBF58476D1CE4E5B9)
            z = (z ^ z >> c(27)) * c(0x94D049BB133111EB)
            s.append(z ^ z >> c(31))

        def rotl(v, k):
            return v << c(k) | v >> c(64 - k)

        for _ in range(count):
            r = rotl(s[1] * c(5), 7) * c(9)
            t = s[1] << c(17)
            s[2] ^= s[0]
            s[3] ^= s[1]
            s[1] ^= s[2]
            s[0] ^= s[3]
            s[2] ^= t
            s[3] = rotl(s[3], 45)
            yield (r >> c(11)).astype(np.float64) * 2.0 ** -53


def _undirected(case, seed):
    """Unique undirected edges (u < v) of the case's graph."""
    if case["kind"] == "rmat":
        a, b, c = RMAT
        s = np.zeros(case["samples"], dtype=np.int64)
        d = s.copy()
        for u in _uniforms(seed, case["samples"], case["scale"]):
            s = s << 1 | (u >= a + b)
            d = d << 1 | ((u >= a) & (u < a + b) | (u >= a + b + c))
    else:
        n = case["n"]
        cdf = np.cumsum((np.arange(n) + case["i0"]) ** (-1.0 / (case["gamma"] - 1.0)))
        cdf /= cdf[-1]
        cdf[-1] = 1.0
        s, d = (np.searchsorted(cdf, u, side="right") for u in _uniforms(seed, case["samples"], 2))
    lo, hi = np.minimum(s, d), np.maximum(s, d)
    keep = lo != hi
    key = np.unique(lo[keep] << 32 | hi[keep])
    return key >> 32, key & 0xFFFFFFFF


def _choose(t, k):
    out = torch.ones_like(t)
    for i in range(k):
        out = out * (t - i)
    return out // math.factorial(k)


class _Lists:
    """Triangles and 4-cliques of an edge list, from rows oriented by (degree, id)."""

    def __init__(self, u, v):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        u, v = (torch.as_tensor(x, dtype=torch.int64, device=dev) for x in (u, v))
        n = int(v.max()) + 1
        self.deg = torch.bincount(torch.cat([u, v]), minlength=n)
        rank = torch.empty_like(self.deg)
        rank[torch.argsort(self.deg, stable=True)] = torch.arange(n, device=dev)
        swap = rank[u] > rank[v]
        a, b = torch.where(swap, rank[v], rank[u]), torch.where(swap, rank[u], rank[v])
        self.n, self.keys = n, torch.sort(a * n + b).values  # a < b in rank
        self.a, self.b = self.keys // n, self.keys % n
        self.ptr = torch.searchsorted(self.a, torch.arange(n + 1, device=dev))
        self.rdeg = torch.empty_like(self.deg)
        self.rdeg[rank] = self.deg

    def edge(self, x, y):
        i = torch.searchsorted(self.keys, x * self.n + y).clamp_(max=len(self.keys) - 1)
        return torch.where(self.keys[i] == x * self.n + y, i, -1)

    def extend(self, rows, step=1 << 23):
        """For row index lists rows[0..m) (one clique each, ranks ascending):
        yields (clique index, next vertex w) with w adjacent to all of them."""
        last = rows[-1]
        size = self.ptr[last + 1] - self.ptr[last]
        ends = torch.cumsum(size, 0)
        total = int(ends[-1]) if len(ends) else 0
        for t0 in range(0, total, step):
            t = torch.arange(t0, min(total, t0 + step), device=last.device)
            c = torch.searchsorted(ends, t, right=True)
            w = self.b[self.ptr[last[c]] + t - (ends[c] - size[c])]
            ok = torch.ones_like(w, dtype=torch.bool)
            for r in rows[:-1]:
                ok &= self.edge(r[c], w) >= 0
            yield c[ok], w[ok]

    def triangles(self):
        found = [(self.a[c], self.b[c], w) for c, w in self.extend([self.a, self.b])]
        return [torch.cat([f[i] for f in found]) for i in range(3)]


def exact(case, seed):
    """Counts of the patterns with a short closed form; None elsewhere, and for
    sgc counts of patterns whose last two vertices are not adjacent (those stop
    a level early and are no subgraph counts)."""
    if case["entry"] not in ("count", "hash", "buffer", "oneshot") or "n_keep" in case or case["samples"] > 1 << 22:
        return None
    pattern, task, _ = _queries(case)[0]
    if task == "sgc" and pattern not in ("triangle", "4clique"):
        return None
    if pattern not in ("triangle", "tailed_triangle", "diamond", "4clique", "4star", "wedge"):
        return None
    g = _Lists(*_undirected(case, seed))
    if pattern in ("wedge", "4star"):
        count = int(_choose(g.deg, 2 if pattern == "wedge" else 3).sum())
    else:
        x, y, z = g.triangles()
        if pattern == "triangle":
            count = len(x)
        elif pattern == "tailed_triangle":
            count = sum(int((g.rdeg[v] - 2).sum()) for v in (x, y, z))
        elif pattern == "diamond":
            per_edge = torch.bincount(torch.cat([g.edge(x, y), g.edge(x, z), g.edge(y, z)]), minlength=1)
            count = int(_choose(per_edge, 2).sum())
        else:
            count = sum(len(w) for _, w in g.extend([x, y, z]))
    out = {"count": _whole(count)}
    if case["entry"] in ("hash", "buffer"):
        out["hash"] = None
    if case["entry"] == "buffer":
        out["matches"] = None
    return out
