"""The work that a user of this framework has it do, as timed cases.

Every case goes through the public Python interface (``beedrill_amd.Context``)
as a user's program does: the graph and, for the learned policy, the network
are resident before the call; a pass is the searches, batch, component run,
graph build or training run itself, with the results read back to the host the
way that program reads them.

Kinds of case
  search      searches of the resident graph one after another (the trial
              loop), each returning its counters; then the last one's depths
              are read.  With check, each is validated with check() and each
              one's depths are read.  Parents are not compared: a vertex
              reached from several vertices of the level before may get any
              of them, so two runs differ; check() is what validates them.
  multi_root  up to 64 searches at once on one graph, every depth row read.
  graphs      many small graphs, searched in one call, depths read.
  components  connected components, labels read.
  build       an edge list in host memory made into the resident graph (CSR,
              search layout, head index), the CSR read back.
  train       the direction network trained from given parameters, and its
              predictions for the samples.
"""
import json
import os

import numpy as np

import beedrill_amd as bd

MODEL = os.path.join(os.path.dirname(bd.__file__), "models", "direction_mlp_32x32.f32")
H = 32  # hidden units of the direction network, both layers
LR = 3e-3  # train_policy's learning rate


def listed():
    return [
        # the smallest call: one search of a small graph, all latency
        {"name": "search_s10", "kind": "search", "graph": "rmat", "scale": 10, "ef": 16,
         "roots": 1, "policy": "beamer", "check": False},
        # a small graph as the tests and the CLI use, validated (--check_results)
        {"name": "checked_s16", "kind": "search", "graph": "rmat", "scale": 16, "ef": 16,
         "roots": 8, "policy": "beamer", "check": True},
        # an ordinary trial loop
        {"name": "trials_s20", "kind": "search", "graph": "rmat", "scale": 20, "ef": 16,
         "roots": 16, "policy": "beamer", "check": False},
        # the benchmark: 64 roots of RMAT scale 24 under the learned policy
        {"name": "trials_s24", "kind": "search", "graph": "rmat", "scale": 24, "ef": 16,
         "roots": 64, "policy": "learned", "check": False},
        # no hubs and an odd number of vertices
        {"name": "trials_er", "kind": "search", "graph": "er", "nv": 3000001, "edges": 40000000,
         "roots": 8, "policy": "beamer", "check": False},
        # thousands of levels with small frontiers
        {"name": "lattice_deep", "kind": "search", "graph": "lattice", "rows": 701, "cols": 1024,
         "roots": 1, "policy": "beamer", "check": False},
        # 64 roots at once, every depth row read
        {"name": "roots64_s18", "kind": "multi_root", "scale": 18, "ef": 16, "roots": 64},
        # a batch of small uneven graphs
        {"name": "graphs_96", "kind": "graphs", "graphs": 96, "lo": 8, "hi": 12},
        # connected components, an ordinary graph and a large one
        {"name": "components_s18", "kind": "components", "scale": 18, "ef": 16},
        {"name": "components_s23", "kind": "components", "scale": 23, "ef": 16},
        # a graph built from a host edge list, odd sizes
        {"name": "build_3m", "kind": "build", "nv": 300007, "edges": 3000017},
        # the direction network trained on a data set of train_policy's size
        {"name": "train_3038", "kind": "train", "samples": 3038, "epochs": 32},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("search", "search", "search", "er", "lattice", "multi_root", "graphs",
                       "components", "build", "train"))
    if kind == "search":
        scale = rng.randint(9, 23)
        return {"kind": "search", "graph": "rmat", "scale": scale, "ef": rng.randint(6, 18),
                "roots": rng.randint(1, 8 if scale > 21 else 20),
                "policy": rng.choice(("beamer", "beamer", "learned", "td_only", "remote_writes_hybrid")
                                     if scale < 21 else ("beamer", "learned")),
                "check": scale < 20 and rng.random() < 0.3}
    if kind == "er":
        nv = _log(rng, 1000, 4000000)
        return {"kind": "search", "graph": "er", "nv": nv, "edges": nv * rng.randint(4, 12),
                "roots": rng.randint(1, 12), "policy": "beamer", "check": False}
    if kind == "lattice":
        return {"kind": "search", "graph": "lattice", "rows": _log(rng, 30, 900),
                "cols": _log(rng, 30, 900), "roots": 1, "policy": "beamer", "check": False}
    if kind == "multi_root":
        return {"kind": "multi_root", "scale": rng.randint(11, 18), "ef": rng.randint(6, 18),
                "roots": rng.randint(5, 64)}
    if kind == "graphs":
        lo = rng.randint(6, 9)
        return {"kind": "graphs", "graphs": rng.randint(7, 150), "lo": lo,
                "hi": lo + rng.randint(1, 3)}
    if kind == "components":
        return {"kind": "components", "scale": rng.randint(12, 22), "ef": rng.randint(3, 18)}
    if kind == "build":
        nv = _log(rng, 2000, 400000)
        return {"kind": "build", "nv": nv, "edges": nv * rng.randint(3, 10) + rng.randint(0, 99)}
    return {"kind": "train", "samples": _log(rng, 300, 3000), "epochs": rng.randint(8, 32)}


def _kronecker(r, scale, m):
    """m edges of a power-law graph of 2^scale vertices (A/B/C/D .57/.19/.19/.05)."""
    s = np.zeros(m, np.int64)
    d = np.zeros(m, np.int64)
    for _ in range(scale):
        q = r.random(m)
        s = 2 * s + (q >= 0.76)
        d = 2 * d + (((q >= 0.57) & (q < 0.76)) | (q >= 0.95))
    return s, d


def _graph(ctx, case, seed):
    if case["graph"] == "rmat":
        ctx.generate_rmat(case["scale"], case["ef"], seed=seed)
    elif case["graph"] == "er":
        ctx.generate_er(case["nv"], case["edges"], seed=seed)
    else:
        ctx.generate_lattice(case["rows"], case["cols"], seed=seed)


def _network(ctx):
    """The shipped direction network with its margin, as the benchmark loads it."""
    ctx.mlp_set(np.fromfile(MODEL, np.float32), H, H)
    with open(os.path.splitext(MODEL)[0] + ".json") as f:
        ctx.set_tuning(learned_margin_milli=int(json.load(f)["margin_milli"]))


def _union(case, seed):
    """The batch's graphs as one edge list, their bounds and a root of each
    (the sizes are the case's, the edges the seed's)."""
    sizes = np.random.default_rng([case["graphs"], case["lo"], case["hi"]])
    r = np.random.default_rng(seed)
    src, dst, vbase, roots = [], [], [0], []
    for _ in range(case["graphs"]):
        scale = int(sizes.integers(case["lo"], case["hi"] + 1))
        nv = int(sizes.integers((1 << scale) * 3 // 4, (1 << scale) + 1))
        s, d = _kronecker(r, scale, nv * int(sizes.integers(8, 25)))
        p = r.permutation(1 << scale)
        s, d = p[s] % nv, p[d] % nv
        keep = s != d
        s, d = s[keep], d[keep]
        roots.append(int(s[0]))
        src.append(s + vbase[-1])
        dst.append(d + vbase[-1])
        vbase.append(vbase[-1] + nv)
    return (np.concatenate(src), np.concatenate(dst), np.array(vbase, np.int64),
            np.array(roots, np.int64))


def _samples(case, seed):
    """Step features and log2 step costs like a training run's, and start parameters."""
    r = np.random.default_rng(seed)
    n = case["samples"]
    x = r.random((n, 8)).astype(np.float32)
    x[:, 7] = r.random(n) < 0.5
    t = (3 + 6 * x[:, 1:2] * r.random((n, 2)) + r.standard_normal((n, 2))).astype(np.float32)
    mask = (r.random((n, 2)) < 0.8).astype(np.float32)
    p = np.zeros(H * 8 + H + H * H + H + 2 * H + 2, np.float32)
    w1, w2, w3 = H * 8, H * 8 + H + H * H, H * 8 + H + H * H + H + 2 * H
    p[:w1] = r.uniform(-1, 1, w1) * np.sqrt(6 / 8)
    p[w1 + H:w2] = r.uniform(-1, 1, H * H) * np.sqrt(6 / H)
    p[w2 + H:w3] = r.uniform(-1, 1, 2 * H) * np.sqrt(6 / H)
    return x, t, mask, p


def prepare(case, seed):
    ctx = bd.Context(0)
    st = {"case": case, "ctx": ctx}
    kind = case["kind"]
    if kind == "search":
        _graph(ctx, case, seed)
        if case["policy"] == "learned":
            _network(ctx)
        if case["graph"] == "lattice":  # one graph whatever the seed: the seed picks the root
            st["roots"] = [int(np.random.default_rng(seed).integers(case["rows"] * case["cols"]))]
        else:
            st["roots"] = [int(v) for v in ctx.pick_roots(case["roots"])]
    elif kind == "multi_root":
        ctx.generate_rmat(case["scale"], case["ef"], seed=seed)
        st["roots"] = ctx.pick_roots(case["roots"])
    elif kind == "graphs":
        src, dst, st["vbase"], st["roots"] = _union(case, seed)
        ctx.from_edges(int(st["vbase"][-1]), src, dst)
    elif kind == "components":
        ctx.generate_rmat(case["scale"], case["ef"], seed=seed)
    elif kind == "build":
        r = np.random.default_rng(seed)
        scale = max(1, (case["nv"] - 1).bit_length())
        s, d = _kronecker(r, scale, case["edges"])
        p = r.permutation(1 << scale)
        st["src"], st["dst"] = p[s] % case["nv"], p[d] % case["nv"]
    else:
        st["x"], st["t"], st["mask"], st["p"] = _samples(case, seed)
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "search":
        stats, depths = [], []
        for i, root in enumerate(st["roots"]):
            r = ctx.bfs(root, policy=case["policy"])
            ok = ctx.check(root) if case["check"] else True
            stats.append((r["source"], r["steps"], r["td_steps"], r["bu_steps"], r["reached"],
                          r["traversed_edges"], ok))
            if case["check"] or i == len(st["roots"]) - 1:
                depths.append(ctx.fetch(depth=True, parent=False)[0])
        return {"stats": np.array(stats, np.int64), "depths": depths}
    if kind == "multi_root":
        depth, _, levels = ctx.multi_root(st["roots"])
        return {"depth": depth, "levels": levels}
    if kind == "graphs":
        depth, _ = ctx.multi_graph(st["vbase"], st["roots"])
        return {"depth": depth}
    if kind == "components":
        r = ctx.components()
        return {"labels": ctx.component_labels(), "components": r["num_components"]}
    if kind == "build":
        ctx.from_edges(case["nv"], st["src"], st["dst"])
        off, cols = ctx.csr()
        return {"off": off, "cols": cols}
    ctx.mlp_set(st["p"], H, H)
    loss = ctx.mlp_train(st["x"], st["t"], st["mask"], epochs=case["epochs"], lr=LR)
    params, _, _ = ctx.mlp_get()
    return {"loss": loss, "params": params, "predicted": ctx.mlp_infer(st["x"], mfma=False)}


def work(case):
    """Bytes: a search reads the bounds of each vertex's list and one
    neighbour, and writes its parent (16 B a vertex); a check reads the whole
    adjacency; a batch of searches reads the adjacency once and writes its
    depth rows; components read the adjacency and write the labels; a build
    reads the edges and writes both directions of each.  Training: three
    products per layer (forward, weights, inputs) and epoch."""
    kind = case["kind"]
    if kind == "search":
        if case["graph"] == "rmat":
            nv, m = 1 << case["scale"], case["ef"] << case["scale"]
        elif case["graph"] == "er":
            nv, m = case["nv"], case["edges"]
        else:
            nv = case["rows"] * case["cols"]
            m = 2 * nv
        adj = 8 * nv + 8 * m
        return {"bytes": case["roots"] * (16 * nv + (adj if case["check"] else 0)) +
                8 * nv * (case["roots"] if case["check"] else 1), "flops": 0}
    if kind == "multi_root":
        nv = 1 << case["scale"]
        return {"bytes": (8 + 4 * case["roots"]) * nv + (8 * case["ef"] << case["scale"]),
                "flops": 0}
    if kind == "graphs":
        nv = case["graphs"] * sum(0.875 * (1 << s) for s in range(case["lo"], case["hi"] + 1)) / (
            case["hi"] - case["lo"] + 1)
        return {"bytes": 20 * nv + 8 * 16 * nv, "flops": 0}  # bounds are checked: every edge read
    if kind == "components":
        nv = 1 << case["scale"]
        return {"bytes": 16 * nv + (8 * case["ef"] << case["scale"]), "flops": 0}
    if kind == "build":
        return {"bytes": (16 + 8) * case["edges"] + 8 * case["nv"], "flops": 0}
    macs = H * 8 + H * H + 2 * H
    return {"bytes": 4 * 12 * case["samples"],
            "flops": 2.0 * macs * case["samples"] * (3 * (case["epochs"] + 1) + 1)}


def _split(p):
    out, at = [], 0
    for shape in ((H, 8), (H,), (H, H), (H,), (2, H), (2,)):
        n = int(np.prod(shape))
        out.append(p[at:at + n].reshape(shape))
        at += n
    return out


def exact(case, seed):
    """The training run in 64 bits; the graph cases return whole numbers only."""
    if case["kind"] != "train":
        return None
    x, t, mask, p = (np.asarray(a, np.float64) for a in _samples(case, seed))
    count = mask.sum()

    def forward(p):
        w1, b1, w2, b2, w3, b3 = _split(p)
        a1 = np.maximum(x @ w1.T + b1, 0)
        a2 = np.maximum(a1 @ w2.T + b2, 0)
        return a1, a2, a2 @ w3.T + b3

    def loss_grad(p):
        w1, b1, w2, b2, w3, b3 = _split(p)
        a1, a2, y = forward(p)
        e = y - t
        dy = 2 * mask * e / count
        d2 = (dy @ w3) * (a2 > 0)
        d1 = (d2 @ w2) * (a1 > 0)
        g = [d1.T @ x, d1.sum(0), d2.T @ a1, d2.sum(0), dy.T @ a2, dy.sum(0)]
        return (mask * e * e).sum() / count, np.concatenate([v.ravel() for v in g])

    m, v = np.zeros_like(p), np.zeros_like(p)
    for k in range(1, case["epochs"] + 1):
        _, g = loss_grad(p)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - LR * (m / (1 - 0.9 ** k)) / (np.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
    return {"loss": float(loss_grad(p)[0]), "params": p, "predicted": forward(p)[2]}
