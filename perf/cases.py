"""Performance cases: the calls a user of this framework makes, over the
ranges they are made in.

  listed()            the named cases, each with what it stands for
  draw(rng)           one more case of the same ranges
  prepare(case, seed) what a program has in hand before the call
  run(state)          one pass through the public entry points
  work(case)          bytes and flops that a pass cannot do without
  exact(case, seed)   the computed numbers in 64 bits (whole numbers: None)

Graph sizes follow the test suite and the benchmark's workloads (G(n, p),
R-MAT with quadrants (0.57, 0.19, 0.19, 0.05), Chung-Lu with planted
communities, batches of the G(n, p) family), scaled so that a graph is made
in well under a second.
"""
import math

import numpy as np

import rdmce_amd as R
from rdmce_amd.learned import NFEAT, CostModel
from rdmce_amd.workloads import expected_er_cliques

H1 = H2 = 32  # hidden widths of the cost model


def listed():
    return [
        # One call on a small graph, upload and release included: what
        # BkSolverWrapper does.  Latency, allocations and launches.
        {"name": "solve_small", "kind": "solve", "graph": "er", "n": 200, "p": 0.1, "pack": False, "lists": False},
        # The same with the cliques themselves asked for.
        {"name": "solve_lists", "kind": "solve", "graph": "er", "n": 1000, "p": 0.02, "pack": False, "lists": True},
        # A resident sparse graph enumerated again and again (a serving loop):
        # the packed search replayed as a captured graph.
        {"name": "replay_sparse", "kind": "plan", "graph": "er", "n": 2048, "p": 0.008, "pack": True, "replay": True,
         "vertex": False, "roots": "all", "param": 0, "stats": False},
        # The plain kernel on a dense random graph: wide roots, deep trees,
        # the bitmap tiers and sharing between wavefronts.
        {"name": "plain_dense", "kind": "plan", "graph": "er", "n": 300, "p": 0.4, "pack": False, "replay": False,
         "vertex": False, "roots": "all", "param": 0, "stats": False},
        # The labelling run of the learned schedule: every 16th edge root of a
        # skewed graph, plain kernel, per-root statistics.
        {"name": "plain_label", "kind": "plan", "graph": "rmat", "scale": 14, "ef": 16, "pack": False,
         "replay": False, "vertex": False, "roots": "stride", "param": 16, "stats": True},
        # Vertex roots (the reference's LEVEL_1) on a graph with communities.
        {"name": "plain_vertex", "kind": "plan", "graph": "cl", "n": 20000, "comm": 20, "p_in": 0.6, "pack": False,
         "replay": False, "vertex": True, "roots": "all", "param": 0, "stats": False},
        # The packed search on a whole skewed graph: a few roots hold most of
        # the tree (the shape of the benchmark's scale-20 workload).
        {"name": "pack_skewed", "kind": "plan", "graph": "rmat", "scale": 14, "ef": 14, "pack": True,
         "replay": False, "vertex": False, "roots": "all", "param": 0, "stats": False},
        # The packed search on the roots below a core bound (the shape of the
        # benchmark's scale-24 workload): many small roots, builds dominate.
        {"name": "pack_core", "kind": "plan", "graph": "rmat", "scale": 18, "ef": 16, "pack": True,
         "replay": False, "vertex": False, "roots": "core", "param": 120, "stats": False},
        # The packed search on a power-law graph with dense communities (the
        # benchmark's Chung-Lu workload): small roots, search dominates.
        {"name": "pack_communities", "kind": "plan", "graph": "cl", "n": 200000, "comm": 100, "p_in": 0.6,
         "pack": True, "replay": False, "vertex": False, "roots": "all", "param": 0, "stats": False},
        # Many independent graphs in one replayed launch.
        {"name": "batch_replay", "kind": "batch", "count": 400, "nmax": 512, "cap": 1e5, "pack": True,
         "replay": True},
        # Training the cost model (forward, backward, Adam).
        {"name": "cost_train", "kind": "train", "n": 20000, "epochs": 6, "batch": 1024},
        # Predicting the cost of every root of a graph.
        {"name": "cost_predict", "kind": "predict", "n": 300000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_er(rng, sparse):
    if sparse:
        n = _log_int(rng, 30, 6000)
        return {"graph": "er", "n": n, "p": round(min(0.5, rng.uniform(4, 24) / n), 6)}
    while True:
        n, p = rng.randint(60, 700), round(rng.uniform(0.05, 0.5), 3)
        if 1e3 <= expected_er_cliques(n, p) <= 2e6:
            return {"graph": "er", "n": n, "p": p}


def _draw_rmat(rng):
    return {"graph": "rmat", "scale": rng.randint(10, 13), "ef": rng.randint(6, 15)}


def _draw_cl(rng):
    n = _log_int(rng, 8000, 120000)
    return {"graph": "cl", "n": n, "comm": max(2, n // rng.randint(1000, 3000)), "p_in": round(rng.uniform(0.4, 0.6), 2)}


def draw(rng):
    kind = rng.choice(["solve", "plan", "plan", "plan", "batch", "train", "predict"])
    if kind == "solve":
        return {"kind": kind, "pack": rng.random() < 0.5, "lists": rng.random() < 0.3, **_draw_er(rng, True)}
    if kind == "plan":
        shape = rng.choice(["sparse", "dense", "rmat", "core", "cl"])
        c = {"kind": kind, "pack": rng.random() < 0.6, "replay": rng.random() < 0.3,
             "vertex": shape != "core" and rng.random() < 0.2, "roots": "all", "param": 0,
             "stats": rng.random() < 0.3}
        if shape in ("sparse", "dense"):
            return {**c, **_draw_er(rng, shape == "sparse")}
        if shape == "rmat":
            if rng.random() < 0.5:
                c.update(roots="stride", param=rng.randint(2, 16))
            return {**c, **_draw_rmat(rng)}
        if shape == "core":
            c.update(roots="core", param=rng.randint(30, 120))
            return {**c, "graph": "rmat", "scale": rng.randint(14, 17), "ef": rng.randint(8, 16)}
        return {**c, **_draw_cl(rng)}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(20, 400), "nmax": rng.randint(64, 512),
                "cap": float(_log_int(rng, 10000, 100000)), "pack": rng.random() < 0.6, "replay": rng.random() < 0.6}
    if kind == "train":
        return {"kind": kind, "n": _log_int(rng, 500, 20000), "epochs": rng.randint(2, 6),
                "batch": rng.choice([256, 500, 1024, 2048])}
    return {"kind": kind, "n": _log_int(rng, 1000, 300000)}


# -- inputs -----------------------------------------------------------------
def _graph(case, seed):
    if case["graph"] == "er":
        g = R.Graph.erdos_renyi(case["n"], case["p"], seed)
    elif case["graph"] == "rmat":
        g = R.Graph.rmat(case["scale"], case["ef"], 0.57, 0.19, 0.19, seed=seed)
    else:
        g = R.Graph.chung_lu_planted(case["n"], 2.1, 20.0, case["comm"], 50, 200, case["p_in"], seed)
    g.SortByOrder(R.OrderType.DEG)
    return g


def _root_order(case, g):
    """Dispatch list of the plan: None = every root, high core first."""
    if case["roots"] == "all":
        return None
    if case["roots"] == "stride":
        return np.arange(0, g.GetNumEdges(), case["param"], dtype=np.uint64)[::-1].copy()
    core = g.GetCoreNumbers()
    v0 = (g.roots(R.ROOT_EDGE) >> np.uint64(32)).astype(np.int64)
    end = int(np.searchsorted(core[v0], case["param"], side="right"))
    return np.arange(end, dtype=np.uint64)[::-1].copy()


def _batch_graphs(case, seed):
    graphs, i = [], 0
    while len(graphs) < case["count"]:
        n, p, s = R.batch_graph_params(seed, i, 32, case["nmax"], 0.05, 0.5)
        i += 1
        if expected_er_cliques(n, p) > case["cap"]:
            continue
        g = R.Graph.erdos_renyi(n, p, s)
        g.SortByOrder(R.OrderType.DEG)
        graphs.append(g)
    return graphs


def _samples(n, seed):
    """Features as mce_root_features gives them (log degrees, core ratios,
    log candidate-set size and its square), and log costs that follow them."""
    rng = np.random.default_rng(seed)
    d0, d1 = 1 + 20 * rng.pareto(1.5, n), 1 + 40 * rng.pareto(1.3, n)
    c0 = rng.random(n)
    c1 = c0 + (1 - c0) * rng.random(n)
    o0, o1 = d0 * rng.random(n), d1 * rng.random(n)
    lt = np.log1p(np.floor(np.minimum(o0, o1) * rng.random(n)))
    x = np.stack([np.log1p(d0), np.log1p(d1), c0, c1, np.log1p(o0), np.log1p(o1), lt, lt * lt], 1)
    y = 7.0 + 0.5 * x[:, 1] + 0.8 * lt + 0.12 * lt * lt + 0.3 * rng.standard_normal(n)
    return np.ascontiguousarray(x, dtype=np.float32), y.astype(np.float32)


def _model_params(x, seed):
    """Initial weights (He-uniform, zero biases) and the standardisation of x."""
    rng = np.random.default_rng(seed + 1)
    layers = []
    for fan_in, fan_out in ((NFEAT, H1), (H1, H2), (H2, 1)):
        lim = math.sqrt(6.0 / fan_in)
        layers += [rng.uniform(-lim, lim, fan_in * fan_out), np.zeros(fan_out)]
    mean = x.mean(0, dtype=np.float64)
    istd = 1.0 / np.sqrt(np.maximum(x.var(0, dtype=np.float64), 1e-12))
    return np.concatenate(layers + [mean, istd]).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "solve":
        st["graph"] = _graph(case, seed)
    elif kind == "plan":
        g = _graph(case, seed)
        st["plan"] = R.Plan(g, pack=case["pack"], use_graph=case["replay"], want_root_stats=case["stats"],
                            root_mode=R.ROOT_VERTEX if case["vertex"] else R.ROOT_EDGE,
                            root_order=_root_order(case, g) if not case["vertex"] else None)
    elif kind == "batch":
        st["batch"] = R.Batch(_batch_graphs(case, seed), pack=case["pack"], use_graph=case["replay"])
    else:
        st["x"], st["y"] = _samples(case["n"], seed)
        st["params"] = _model_params(st["x"], seed)
        st["model"] = CostModel(seed)
        if kind == "predict":
            st["model"].set_params(st["params"])
    return st


# -- the pass -----------------------------------------------------------------
def _padded(a, n):
    """`a` with zeros up to n entries: graphs of one case differ in size."""
    if len(a) > n:
        raise ValueError(f"{len(a)} entries, room for {n}")
    res = np.zeros((n,) + np.shape(a)[1:], dtype=np.asarray(a).dtype)
    res[:len(a)] = a
    return res


def _cliques(case, out):
    n, m = _edges(case)
    res = {"totals": np.array([out.count, out.hash, out.total_nodes, out.search_bytes], dtype=np.uint64),
           "hist": _padded(out.hist, 4096)}
    if out.cliques is not None:  # in any order from the library: sorted
        cl = sorted(out.cliques)
        cap = int(4 * m) + 4096  # sparse graphs: about one clique per edge
        res["sizes"] = _padded(np.array([len(c) for c in cl], dtype=np.int64), cap)
        res["members"] = _padded(np.array([v for c in cl for v in c], dtype=np.int64), 4 * cap)
    if out.root_nodes is not None:
        res["root_nodes"] = _padded(out.root_nodes, int(1.5 * n if case.get("vertex") else 1.5 * m) + 1024)
    return res


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "solve":
        return _cliques(case, R.solve(state["graph"], pack=case["pack"], want_list=case["lists"]))
    if kind == "plan":
        return _cliques(case, state["plan"].run())
    if kind == "batch":
        out = state["batch"].run()
        return {"count": out.count, "hash": out.hash, "hist": _padded(out.hist.T, 640).T,
                "totals": np.array([out.total_count, out.total_nodes], dtype=np.uint64)}
    model = state["model"]
    if kind == "train":
        model.set_params(state["params"])
        loss = model.train(state["x"], state["y"], epochs=case["epochs"], batch=case["batch"], lr=3e-3, seed=1)
        return {"params": model.params(), "loss": np.array([loss], dtype=np.float32)}
    return model.predict(state["x"])


# -- what a pass cannot do without ------------------------------------------------
def _edges(case):
    if case["graph"] == "er":
        return case["n"], 0.5 * case["n"] * (case["n"] - 1) * case["p"]
    if case["graph"] == "rmat":
        return 0.7 * 2 ** case["scale"], 0.9 * case["ef"] * 2 ** case["scale"]
    return case["n"], 10.0 * case["n"] + case["comm"] * 0.5 * 125 ** 2 * case["p_in"]


def work(case):
    """Enumeration: the CSR (8 B per vertex, 4 B per entry) read once and the
    histogram written; how much set work the tree takes is known only once it
    has been enumerated, so no flops are claimed.  Cost model: samples and
    weights read, results written; multiply-adds of the three layers (a
    training step has three such products, one forward and two backward)."""
    kind = case["kind"]
    if kind in ("solve", "plan"):
        n, m = _edges(case)
        return {"bytes": int(8 * n + 8 * m + 512), "flops": 0}
    if kind == "batch":
        m = case["count"] * 0.25 * (case["nmax"] / 2) ** 2 * 0.2
        return {"bytes": int(8 * case["count"] * case["nmax"] / 2 + 8 * m + 600 * case["count"]), "flops": 0}
    mac = NFEAT * H1 + H1 * H2 + H2
    if kind == "train":
        steps = case["n"] * case["epochs"]
        return {"bytes": int(4 * (NFEAT + 1) * case["n"]), "flops": int(3 * 2 * mac * steps)}
    return {"bytes": int(4 * (NFEAT + 1) * case["n"]), "flops": int(2 * mac * case["n"])}


# -- the same numbers in 64 bits --------------------------------------------------
_M64 = (1 << 64) - 1


def _mix(x):
    z = (x + 0x9E3779B97F4A7C15) & _M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    return z ^ (z >> 31)


def _shuffled(n, seed, epoch):
    """The epoch's sample order: Fisher-Yates with xoshiro256**."""
    x = _mix(seed ^ _mix((epoch + 0x632BE59BD9B4E019) & _M64))
    s = []
    for _ in range(4):
        s.append(_mix(x))
        x = (x + 0x9E3779B97F4A7C15) & _M64
    rot = lambda v, k: ((v << k) | (v >> (64 - k))) & _M64  # noqa: E731
    idx = list(range(n))
    for i in range(n - 1, 0, -1):
        bound = i + 1
        while True:
            r = (rot((s[1] * 5) & _M64, 7) * 9) & _M64
            t = (s[1] << 17) & _M64
            s[2] ^= s[0]
            s[3] ^= s[1]
            s[1] ^= s[2]
            s[0] ^= s[3]
            s[2] ^= t
            s[3] = rot(s[3], 45)
            lo = (r * bound) & _M64
            if lo >= bound or lo >= ((1 << 64) - bound) % bound:
                break
        j = (r * bound) >> 64
        idx[i], idx[j] = idx[j], idx[i]
    return np.array(idx)


def _split(p):
    sizes = [NFEAT * H1, H1, H1 * H2, H2, H2, 1, NFEAT, NFEAT]
    w1, b1, w2, b2, w3, b3, mean, istd = np.split(p, np.cumsum(sizes)[:-1])
    return w1.reshape(NFEAT, H1), b1, w2.reshape(H1, H2), b2, w3, b3, mean, istd


def _forward(p, x):
    w1, b1, w2, b2, w3, b3, mean, istd = _split(p)
    xn = (x - mean) * istd
    h1 = np.maximum(xn @ w1 + b1, 0.0)
    h2 = np.maximum(h1 @ w2 + b2, 0.0)
    return xn, h1, h2, h2 @ w3 + b3[0]


def exact(case, seed):
    if case["kind"] not in ("train", "predict"):
        return None  # whole numbers
    x, y = _samples(case["n"], seed)
    p = _model_params(x, seed).astype(np.float64)
    x, y = x.astype(np.float64), y.astype(np.float64)
    if case["kind"] == "predict":
        return _forward(p, x)[3]
    nt = p.size - 2 * NFEAT
    m, v = np.zeros(nt), np.zeros(nt)
    step, loss = 0, 0.0
    lr, b1, b2, eps = float(np.float32(3e-3)), float(np.float32(0.9)), float(np.float32(0.999)), float(np.float32(1e-8))
    for ep in range(case["epochs"]):
        idx = _shuffled(case["n"], 1, ep)
        loss = 0.0
        for at in range(0, case["n"], case["batch"]):
            rows = idx[at:at + case["batch"]]
            xn, h1, h2, out = _forward(p, x[rows])
            w2, w3 = _split(p)[2], _split(p)[4]
            d = out - y[rows]
            loss += float(d @ d)
            dy = 2.0 * d / len(rows)
            d2 = np.where(h2 > 0, dy[:, None] * w3, 0.0)
            d1 = np.where(h1 > 0, d2 @ w2.T, 0.0)
            g = np.concatenate([(xn.T @ d1).ravel(), d1.sum(0), (h1.T @ d2).ravel(), d2.sum(0), h2.T @ dy,
                                [dy.sum()]])
            step += 1
            m = b1 * m + (1 - b1) * g
            v = b2 * v + (1 - b2) * g * g
            p[:nt] -= lr * (m / (1 - b1 ** step)) / (np.sqrt(v / (1 - b2 ** step)) + eps)
    return {"params": p, "loss": np.array([loss / case["n"]])}
