"""The work a user has this framework do, as cases a timing program can run.

Every case goes through the package's public entry points (the Python binding
of libmce.so). Graph sizes are those of the repository's own configurations,
tests and benchmark, or generic ones between them:

  run     one whole call on a host graph: upload, order, count, destroy
  step    a graph resident on the GPU: degeneracy ordering + enumeration, the
          benchmark's step
  batch   one whole run_batch call on a packed batch of graphs
  noalloc ordering + the allocation-free count on a resident graph
  order   ordering + orientation of a resident graph, and the ordering copied
          back as priority and split arrays
  grad    full-batch forward and backward pass of the cost model

All enumeration outputs are whole numbers; the cost model's are float32.
"""
import importlib.util
import math
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _engine():
    if "mce_gpu_amd" not in sys.modules:
        path = os.path.join(ROOT, "mce-gpu_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location("mce_gpu_amd", path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["mce_gpu_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["mce_gpu_amd"]


def _model(family):
    return os.path.join(ROOT, "mce-gpu_amd", f"cost_model_{family}.mlp")


def listed():
    return [
        # one small graph from a program's memory: all latency
        dict(name="run_er300", op="run", graph="er", n=300, m=1800, level=1, induced=1, worklist=1),
        # Erdos-Renyi 4096, the small configuration with the plain method
        dict(name="step_er4096_ip", op="step", graph="er", n=4096, m=65536, level=1, induced=1, worklist=1),
        # a power-law graph of 0.6 M cliques by arc subproblems (-p l2 -i px -w wl)
        dict(name="step_rmat12_l2", op="step", graph="rmat", scale=12, ef=16, level=2, induced=2, worklist=2),
        # a power-law graph of 1e8 cliques in few heavy subproblems (-p l1 -i px -w wl)
        dict(name="step_rmat14_wl", op="step", graph="rmat", scale=14, ef=16, level=1, induced=2, worklist=2),
        # the same family without induced outside rows (-p l1 -i p -w wl)
        dict(name="step_rmat13_ip", op="step", graph="rmat", scale=13, ef=11, level=1, induced=1, worklist=2),
        # social-network-like graph of the large configuration's family, learned schedule
        dict(name="step_cl18_learned", op="step", graph="cl", n=262144, planted=128, level=1, induced=2, worklist=3,
             learned=True),
        # the same family, an odd size, plain schedule
        dict(name="step_cl30011", op="step", graph="cl", n=30011, planted=14, level=1, induced=2, worklist=2,
             learned=False),
        # 1/64 of the benchmark's batch of block-model graphs, as it runs them
        dict(name="batch_sbm64", op="batch", graphs=64, n_min=64, n_max=4096, p_in=0.3, p_out=0.01, worklist=3,
             learned=True),
        # many small graphs in one call, default settings
        dict(name="batch_sbm_small", op="batch", graphs=301, n_min=64, n_max=300, p_in=0.3, p_out=0.01, worklist=1,
             learned=False),
        # one dense block-model graph in a program that may not allocate
        dict(name="noalloc_sbm1500", op="noalloc", n=1500, p_in=0.3, p_out=0.01, induced=2),
        # the ordering alone of a large sparse graph (Table 1's first column)
        dict(name="order_rmat18", op="order", graph="rmat", scale=18, ef=16),
        # one training gradient of the cost model over labelled subproblems
        dict(name="grad_100k", op="grad", rows=100003),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "er", "rmat", "rmat", "cl", "cl", "batch", "batch", "noalloc", "order", "grad"])
    if kind == "run":
        n = _log(rng, 200, 5000)
        return dict(op="run", graph="er", n=n, m=n * rng.randint(4, 16), level=rng.choice([1, 2]),
                    induced=rng.choice([1, 2]), worklist=rng.choice([1, 2]))
    if kind == "er":
        n = _log(rng, 1000, 50000)
        return dict(op="step", graph="er", n=n, m=n * rng.randint(4, 16) + rng.randint(0, 99), level=rng.choice([1, 2]),
                    induced=rng.choice([1, 2]), worklist=rng.choice([1, 2]))
    if kind == "rmat":
        level, induced = rng.choice([(1, 2), (1, 2), (2, 2), (1, 1)])
        scale = rng.randint(10, {(1, 2): 14, (2, 2): 12, (1, 1): 13}[level, induced])
        return dict(op="step", graph="rmat", scale=scale, ef=rng.randint(6, 11 if scale > 12 and induced == 1 else 16),
                    level=level, induced=induced, worklist=rng.choice([1, 2]) if scale < 13 else 2)
    if kind == "cl":
        n = _log(rng, 4000, 262144)
        return dict(op="step", graph="cl", n=n, planted=n >> 11, level=1, induced=2, worklist=rng.choice([2, 3]),
                    learned=rng.choice([False, True]))
    if kind == "batch":
        n_max = _log(rng, 200, 4096)
        most = 301 if n_max <= 600 else max(2, min(64, int(64 * (4096 / n_max) ** 2)))
        return dict(op="batch", graphs=_log(rng, 1, most), n_min=64, n_max=n_max, p_in=0.3, p_out=0.01,
                    worklist=rng.choice([1, 2, 3]), learned=rng.choice([False, True]))
    if kind == "noalloc":
        return dict(op="noalloc", n=_log(rng, 100, 2500), p_in=0.3, p_out=0.01, induced=rng.choice([1, 2]))
    if kind == "order":
        return dict(op="order", graph="rmat", scale=rng.randint(12, 18), ef=rng.randint(4, 16))
    return dict(op="grad", rows=_log(rng, 1000, 200000))


def _graph(m, case, seed):
    if case["graph"] == "er":
        return m.gen_er(case["n"], case["m"], seed)
    if case["graph"] == "rmat":
        return m.gen_rmat(case["scale"], case["ef"], seed=seed)
    return m.gen_chung_lu(case["n"], 2.1, 24.0, case["planted"], 20, 60, seed=seed)


def _count_args(case):
    kw = dict(level=case["level"], induced=case["induced"], worklist=case["worklist"])
    if case.get("learned"):
        kw["model_path"] = _model("cl")
    return kw


def _training_rows(case, seed):
    """Feature rows around the committed model's training statistics and
    labels in the range of log1p(tree nodes)."""
    m = _engine()
    ref = m.mlp_params(m.mlp_load(_model("cl")))
    rng = np.random.default_rng(seed)
    z = rng.standard_normal((case["rows"], m.MLP_FEATURES), dtype=np.float32)
    x = (ref["mu"] + ref["sigma"] * z).astype(np.float32)
    y = np.maximum(0.7, 4.0 + 2.5 * z[:, 1] + rng.standard_normal(case["rows"], dtype=np.float32)).astype(np.float32)
    return x, y, m.mlp_init(x, seed=seed)


def prepare(case, seed):
    m = _engine()
    op = case["op"]
    if op == "grad":
        x, y, model = _training_rows(case, seed)
        return dict(op=op, x=x, y=y, model=model)
    if op == "run":
        return dict(op=op, g=_graph(m, case, seed), kw=_count_args(case))
    if op == "batch":
        off, g = m.gen_sbm_batch(case["graphs"], case["n_min"], case["n_max"], 4, case["p_in"], case["p_out"],
                                 seed=seed)
        kw = dict(level=1, induced=2, worklist=case["worklist"])
        keep = None
        if case["learned"]:
            keep = _model("sbm").encode()
            kw.update(schedule=m.SCHED_LEARNED, model_path=keep)
        return dict(op=op, off=off, g=g, kw=kw, keep=keep)
    if op == "noalloc":
        _, g = m.gen_sbm_batch(1, case["n"], case["n"], 4, case["p_in"], case["p_out"], seed=seed)
        return dict(op=op, dg=m.DeviceGraph(g), kw=dict(induced=case["induced"]))
    dg = m.DeviceGraph(_graph(m, case, seed))
    if op == "order":
        return dict(op=op, dg=dg)
    return dict(op=op, dg=dg, kw=_count_args(case))


def _result(r):
    """A count's whole result as arrays of whole numbers."""
    hist = np.zeros(4098, np.int64)
    for k, v in r["hist"].items():
        hist[k] = v
    keys = ("count", "tree_nodes", "max_clique_size", "degeneracy", "max_degree", "max_out_degree")
    out = {k: int(r[k]) for k in keys}
    out["hash"] = np.array([r["hash"]], np.uint64).view(np.int64)
    out["hist"] = hist
    return out


def run(state):
    m = _engine()
    op = state["op"]
    if op == "grad":
        grad, loss = m.mlp_grad(state["model"], state["x"], state["y"])
        return dict(grad=grad, loss=np.array([loss]))
    if op == "run":
        return _result(m.run(state["g"], **state["kw"]))
    if op == "batch":
        counts, r = m.run_batch(state["off"], state["g"], **state["kw"])
        return dict(_result(r), counts=counts.view(np.int64))
    info = state["dg"].order()
    if op == "order":
        prio, split, _ = state["dg"].download(col=False)
        return dict(degeneracy=info["degeneracy"], max_degree=info["max_degree"],
                    max_out_degree=info["max_out_degree"], prio=prio.astype(np.int64), split=split.view(np.int64))
    if op == "noalloc":
        return _result(state["dg"].count_noalloc(**state["kw"]))
    return _result(state["dg"].count(**state["kw"]))


def _size(case):
    """(vertices, arcs) a case's graph has on average."""
    if case["op"] in ("batch", "noalloc"):
        lo, hi = (case["n_min"], case["n_max"]) if case["op"] == "batch" else (case["n"], case["n"])
        k = case.get("graphs", 1)
        n2 = (hi * hi + hi * lo + lo * lo) / 3.0
        return k * (lo + hi) / 2.0, k * n2 * (case["p_in"] / 4 + case["p_out"] * 3 / 4)
    if case["graph"] == "er":
        return case["n"], 2.0 * case["m"]
    if case["graph"] == "rmat":
        return 2.0 ** case["scale"], 2.0 * case["ef"] * 2 ** case["scale"]
    return case["n"], 24.0 * case["n"]


def work(case):
    if case["op"] == "grad":
        # the rows and labels once; three multiply-adds per weight and row
        weights = 16 * 64 + 64 * 64 + 64
        return dict(bytes=4.0 * 17 * case["rows"], flops=6.0 * weights * case["rows"])
    n, m = _size(case)
    # the ordering reads the CSR (8-byte offsets, 4-byte columns) and writes
    # 4-byte priorities and 8-byte splits; the enumeration reads the CSR once
    # more. Its set operations are integer work and depend on the graph, not
    # on the sizes alone: they are not counted here.
    return dict(bytes=(12.0 * n + (8.0 * n + 4.0 * m) * (1 if case["op"] == "order" else 2)), flops=0.0)


def exact(case, seed):
    """The cost model's gradient and loss in 64 bits; every other output is a
    whole number."""
    if case["op"] != "grad":
        return None
    x, y, model = _training_rows(case, seed)
    p = _engine().mlp_params(model)
    x = (x.astype(np.float64) - p["mu"].astype(np.float64)) / p["sigma"].astype(np.float64)
    w1, w2, w3 = (p[k].astype(np.float64) for k in ("W1", "W2", "w3"))
    h1 = np.maximum(x @ w1 + p["b1"].astype(np.float64), 0)
    h2 = np.maximum(h1 @ w2 + p["b2"].astype(np.float64), 0)
    err = h2 @ w3 + p["b3"] - y.astype(np.float64)
    dy = 2.0 * err / case["rows"]
    d2 = np.where(h2 > 0, dy[:, None] * w3, 0.0)
    d1 = np.where(h1 > 0, d2 @ w2.T, 0.0)
    grad = np.concatenate([(x.T @ d1).ravel(), d1.sum(0), (h1.T @ d2).ravel(), d2.sum(0), h2.T @ dy, [dy.sum()]])
    return dict(grad=grad, loss=np.array([np.mean(err * err)]))
