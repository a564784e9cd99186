"""Performance cases of the incremental graph engine: the calls its users make,
over the sizes they make them at.

Graphs are R-MAT (a, b, c, d = 0.57, 0.19, 0.19, 0.05, ids not permuted,
self-loops and duplicates removed), as in the benchmark; vertex counts that
are no power of two reject the ids beyond them. Updates are deletes drawn
uniformly from the current edges and R-MAT inserts that are not present.

An update case applies a period's batches, reads the result, and takes the
period back with the inverse batches, so that a pass leaves the engine's graph
as it found it. Kinds:
  update  form "call"    Engine.apply_batch with the caller's host records
          form "phases"  Engine.del_edge and Engine.add_edge one after the other
          form "stream"  Engine.load_updates, then apply_next_batches(each=True)
          form "group"   Engine.load_updates, then apply_next_batches as one group
  solve   Engine.init_graph + start: the fixed point from scratch
  query   Engine.query (results in host memory) or, with device, query_noalloc
  serve   Server.submit_update / submit_query, with an HBM edge budget or without
Parents are not returned: any tight in-neighbour is a valid parent, and which
one an engine holds depends on the order of its atomics.
"""
import math

import numpy as np
import torch

import coincgraph_amd as cg

DEV = "cuda" if torch.cuda.is_available() else "cpu"
ABC = (0.57, 0.19, 0.19)
WEIGHT_SEED = 64
BASE = dict(kind="update", algo="sssp", n=65536, ef=16, sym=False, weights="ref128", form="call", staged=False,
            batch=1000, nbatches=1, churn=0.0, k=1, budget=0.0, device=False)


def _case(**kw):
    return dict(BASE, **kw)


def listed():
    return [
        # the smallest calls: one edit each way on a graph of a few thousand vertices (the smoke test's
        # size), deletes and inserts in calls of their own, as the samples make them
        _case(name="sssp_4k_phases", n=4096, batch=500, form="phases"),
        # the benchmark's BFS workload: batches of 1000 + 1000 that arrive one at a time in host memory
        _case(name="bfs_64k_call", algo="bfs"),
        # the benchmark's headline workload: a stream of 100,000 + 100,000 batches on R-MAT scale 22,
        # replayed batch by batch
        _case(name="sssp_4m_stream", n=1 << 22, weights="hash64", form="stream", batch=100_000, nbatches=8),
        # the benchmark's components workload (an undirected graph, large batches of pairs) at a quarter of its size
        _case(name="cc_4m_sym_call", algo="cc", n=1 << 22, ef=8, sym=True, batch=250_000),
        # the benchmark's PageRank workload at an eighth of its size: one large batch each way
        _case(name="pr_4m_call", algo="pr", n=1 << 22, batch=62_500),
        # a first PageRank solve, an odd number of vertices
        _case(name="pr_1m_solve", kind="solve", algo="pr", n=1_000_003),
        # a first shortest-path solve of a large graph
        _case(name="sssp_3m_solve", kind="solve", n=3_000_017, weights="hash64"),
        # a 64-source BFS for a caller that keeps the depths on the device
        _case(name="bfs64_200k_query_device", kind="query", algo="bfs", n=200_003, k=64, device=True),
        # a weighted multi-source query with its distances in host memory
        _case(name="sssp16_1m_query", kind="query", n=1 << 20, weights="hash64", k=16),
        # 64 sources kept current through every batch of a stream
        _case(name="sssp64_256k_stream", n=1 << 18, weights="hash64", form="stream", k=64, batch=6250, nbatches=4),
        # a backlog of ten batches applied as one group; later batches delete some of what earlier ones added
        _case(name="sssp_1m_group", n=1 << 20, form="group", batch=25_000, nbatches=10, churn=0.05),
        # the serving workload in small: update requests and a query through the server, 30% of the edges in HBM
        _case(name="serve_500k_budget", kind="serve", n=500_009, ef=32, weights="hash64", batch=20_000, nbatches=6, k=8,
              budget=0.3),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    weights = rng.choice(["ref128", "hash64"])
    kind = rng.choice(["update", "update", "update", "multi", "solve", "query", "serve"])
    if kind == "update":
        algo = rng.choice(["bfs", "sssp", "sssp", "cc", "pr"])
        n = logint(3000, 2_000_000)
        form = rng.choice(["call", "call", "phases", "stream", "group"])
        nb = rng.randint(2, 8) if form in ("stream", "group") and algo != "pr" else 1
        sym = algo == "cc" and rng.random() < 0.5
        return _case(algo=algo, n=n, ef=rng.choice([8, 16]), sym=sym, weights=weights, form=form,
                     staged=form == "call" and algo != "pr" and rng.random() < 0.3,
                     batch=max(10, int(n * rng.uniform(0.002, 0.03))), nbatches=nb,
                     churn=0.05 if form == "group" else 0.0)
    if kind == "multi":
        n = logint(3000, 300_000)
        return _case(algo=rng.choice(["bfs", "sssp"]), n=n, weights=weights, form=rng.choice(["call", "stream"]),
                     k=rng.choice([2, 7, 16, 33, 64]), batch=max(10, int(n * rng.uniform(0.005, 0.03))),
                     nbatches=rng.randint(1, 4))
    if kind == "solve":
        algo = rng.choice(["bfs", "sssp", "cc", "pr"])
        return _case(kind="solve", algo=algo, n=logint(3000, 3_000_000 if algo != "pr" else 1_000_000),
                     ef=rng.choice([8, 16]), sym=algo == "cc" and rng.random() < 0.5, weights=weights)
    if kind == "query":
        device = rng.random() < 0.5
        return _case(kind="query", algo=rng.choice(["bfs", "sssp"]), n=logint(3000, 500_000 if device else 1_000_000),
                     weights=weights, k=rng.choice([1, 3, 8, 16] if not device else [1, 5, 16, 40, 64]), device=device)
    n = logint(20_000, 500_000)
    return _case(kind="serve", n=n, weights=weights, batch=int(n * rng.uniform(0.005, 0.04)),
                 nbatches=rng.randint(2, 6), k=rng.randint(1, 8), budget=rng.choice([0.0, 0.3]))


# ------------------------------------------------------------------ inputs
def _rmat(gen, n, m):
    """m R-MAT samples (source, destination) below n."""
    scale = max(1, (n - 1).bit_length())
    a, b, c = ABC
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        r = torch.rand(m, generator=gen, device=DEV)
        u = u * 2 + (r >= a + b).long()
        v = v * 2 + (((r >= a) & (r < a + b)) | (r >= a + b + c)).long()
    ok = (u < n) & (v < n) & (u != v)
    return u[ok], v[ok]


def _keys(u, v, n, sym):
    if sym:
        u, v = torch.minimum(u, v), torch.maximum(u, v)
    return u * n + v


def _world(case, seed):
    """Edge keys (u * n + v; one per pair when symmetric) and the batches' (delete, insert) keys."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1_000_003 * int(seed) + case["n"])
    n, sym = case["n"], case["sym"]
    base = torch.unique(_keys(*_rmat(gen, n, case["ef"] * n), n, sym))
    batches = []
    if case["kind"] in ("update", "serve"):
        nb, want = case["nbatches"], case["batch"] * case["nbatches"]
        pool = torch.empty(0, dtype=torch.int64, device=DEV)
        while pool.numel() < want:
            k = _keys(*_rmat(gen, n, 2 * want + 1000), n, sym)
            at = torch.searchsorted(base, k).clamp(max=base.numel() - 1)
            pool = torch.unique(torch.cat([pool, k[base[at] != k]]))
        adds = pool[torch.randperm(pool.numel(), generator=gen, device=DEV)[:want]].view(nb, -1)
        dels = base[torch.randperm(base.numel(), generator=gen, device=DEV)[:want]].view(nb, -1).clone()
        again = int(case["churn"] * case["batch"])
        for b in range(1, nb if again else 0):
            dels[b, :again] = adds[b - 1, :again]
        batches = [(dels[b], adds[b]) for b in range(nb)]
    return base, batches


def _both(key, n, sym):
    u, v = key // n, key % n
    if sym:
        u, v = torch.stack([u, v], 1).reshape(-1), torch.stack([v, u], 1).reshape(-1)
    return u, v


def _records(key, n, sym):
    u, v = _both(key, n, sym)
    return cg.edges_array(u.cpu().numpy(), v.cpu().numpy())


def _csr(key, n, sym):
    u, v = _both(key, n, sym)
    k = torch.sort(u * n + v).values
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(k // n, minlength=n), 0)
    return cg.HostGraph(n, off.cpu().numpy().astype(np.uint64), (k % n).to(torch.int32).cpu().numpy().view(np.uint32))


def _sources(case):
    """Spread over the ids; vertex 0, the largest hub, first."""
    return np.array([i * 65537 % case["n"] for i in range(case["k"])], dtype=np.uint32)


def prepare(case, seed):
    n, sym = case["n"], case["sym"]
    base, batches = _world(case, seed)
    graph = _csr(base, n, sym)
    kw = {}
    if case["algo"] == "pr":
        kw.update(pr_epsilon=1e-7, pr_max_rounds=1000)
    if case["weights"] == "hash64":
        kw.update(weight_mode=cg.WEIGHT_HASH64, weight_seed=WEIGHT_SEED)
    if case["budget"]:
        kw["cache_bytes"] = int(case["budget"] * 2 * 4 * graph.m)  # both directions' rows
    if sym:
        kw["flags"] = cg.CFG_SYMMETRIC
    # a query's engine serves traversal algorithms alike; its own state is not used
    e = cg.Engine(case["algo"], **kw)
    e.load_graph(graph)
    state = {"case": case, "engine": e, "sources": _sources(case)}
    if case["kind"] == "query":
        if case["device"]:
            state["out"] = torch.empty((case["k"], n), dtype=torch.int32, device=DEV)
        return state
    e.init_graph(state["sources"] if case["kind"] == "update" and case["k"] > 1 else 0)
    if case["kind"] == "solve":
        return state
    e.start()
    there = [(_records(d, n, sym), _records(a, n, sym)) for d, a in batches]
    back = [(a, d) for d, a in reversed(there)]
    state["there"], state["back"] = there, back
    if case["form"] in ("stream", "group"):
        every = there + back
        state["stream"] = cg.UpdateStream(np.concatenate([a for _, a in every]), np.concatenate([d for d, _ in every]),
                                          np.array([(len(a), len(d)) for d, a in every], dtype=np.uint32))
    if case["kind"] == "serve":
        state["server"] = cg.Server(e)
    return state


# -------------------------------------------------------------------- runs
def _apply(e, case, batches):
    for dels, adds in batches:
        if case["form"] == "phases":
            e.del_edge(dels)
            e.add_edge(adds)
        else:
            e.apply_batch(dels, adds, staged=case["staged"])


def _submit(server, batches):
    for t in [server.submit_update(dels, adds) for dels, adds in batches]:
        if server.wait(t)["status"] != cg.OK:
            raise RuntimeError("an update request failed")


def run(state):
    case, e = state["case"], state["engine"]
    kind, form = case["kind"], case["form"]
    if kind == "solve":
        e.init_graph(0)
        e.start()
        return e.values()
    if kind == "query":
        if not case["device"]:
            return e.query(case["algo"], state["sources"])
        out = state["out"]
        e.query_noalloc(case["algo"], state["sources"], out.data_ptr(), out.numel() * 4)
        return out
    if kind == "serve":
        server = state["server"]
        _submit(server, state["there"])
        reply = server.wait(server.submit_query(case["algo"], state["sources"]))
        _submit(server, state["back"])
        return reply["result"]
    if form in ("stream", "group"):
        nb = case["nbatches"]
        e.load_updates(state["stream"])
        e.apply_next_batches(nb, each=form == "stream")
        values = e.values()
        e.apply_next_batches(nb, each=form == "stream")
        return values
    _apply(e, case, state["there"])
    values = e.values()
    _apply(e, case, state["back"])
    return values


def work(case):
    """Bytes each pass has to move once: the graph's rows (4 B an edge, a 16-B
    descriptor and an 8-B state word a vertex) where it reads the whole graph,
    12 B an update record and its slot and row descriptor in both directions,
    4 B a result. Traversals do one addition and comparison an edge."""
    n, m = case["n"], case["n"] * case["ef"] * (2 if case["sym"] else 1)
    records = 4 * case["batch"] * case["nbatches"] * (2 if case["sym"] else 1)  # there and back
    results = 4 * n * (case["k"] if case["kind"] in ("query", "serve") or case["algo"] != "pr" else 1)
    whole = 4 * m + 24 * n
    if case["kind"] in ("solve", "query"):
        return {"bytes": whole + results, "flops": 2.0 * m * case["k"]}
    moved = records * (12 + (1 if case["sym"] else 2) * 20) + results
    if case["kind"] == "serve" or case["algo"] == "pr":
        moved += whole
    return {"bytes": moved, "flops": 2.0 * records * case["k"]}


# ------------------------------------------------------- reference results
def _shr(x, k):
    return (x >> k) & ((1 << (64 - k)) - 1)


def _signed(x):
    return x - (1 << 64) if x >= 1 << 63 else x


def _weight(case, u, v):
    if case["algo"] == "bfs":
        return torch.ones_like(u)
    if case["algo"] == "cc":
        return torch.zeros_like(u)
    if case["weights"] == "ref128":
        return (u + v) % 128 + 1
    z = ((u << 32 | v) ^ WEIGHT_SEED) + _signed(0x9E3779B97F4A7C15)
    z = (z ^ _shr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _signed(0x94D049BB133111EB)
    return ((z ^ _shr(z, 31)) & 63) + 1


def _relaxed(value, u, v, w):
    """The fixed point of value[v] <= value[u] + w(u, v)."""
    while True:
        new = value.scatter_reduce(0, v, value[u] + w, "amin")
        if torch.equal(new, value):
            return value
        value = new


def exact(case, seed):
    n, sym, algo = case["n"], case["sym"], case["algo"]
    key, batches = _world(case, seed)
    for dels, adds in batches:
        key = torch.cat([key, adds])
    if batches:
        gone = torch.sort(torch.cat([d for d, _ in batches])).values
        at = torch.searchsorted(gone, key).clamp(max=gone.numel() - 1)
        key = key[gone[at] != key]
    u, v = _both(key, n, sym)
    if algo == "pr":
        deg = torch.bincount(u, minlength=n).double()
        order = torch.sort(v * n + u).values
        rows = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
        rows[1:] = torch.cumsum(torch.bincount(v, minlength=n), 0)
        cols = order % n
        p = torch.sparse_csr_tensor(rows, cols, 0.85 / deg[cols], size=(n, n), dtype=torch.float64, device=DEV)
        x = torch.full((n,), 0.15, dtype=torch.float64, device=DEV)
        for _ in range(400):
            new = 0.15 + (p @ x[:, None])[:, 0]
            done = float((new - x).abs().max()) < 1e-12 * float(new.max())
            x = new
            if done:
                break
        return x.cpu().numpy()
    w = _weight(case, u, v)
    if algo == "cc":
        return _relaxed(torch.arange(n, device=DEV), u, v, w).cpu().numpy().astype(np.uint32)
    inf = 1 << 40
    rows = []
    for s in _sources(case).tolist():
        value = torch.full((n,), inf, dtype=torch.int64, device=DEV)
        value[s] = 0
        value = _relaxed(value, u, v, w)
        rows.append(torch.where(value >= inf, torch.full_like(value, 0xFFFFFFFF), value))
    got = torch.stack(rows).cpu().numpy().astype(np.uint32)
    if case["kind"] == "query" and case["device"]:
        return torch.from_numpy(got.view(np.int32))
    if case["kind"] in ("query", "serve") or case["k"] > 1:
        return got
    return got[0]
