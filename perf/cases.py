"""Timed cases of the engine: what a user's program has it count, by way of
the `tcamd` package, from a file of a few thousand records to R-MAT scale 23.

    listed()            the standing cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what the program holds before the call
    run(state)          one pass
    work(case)          bytes a pass cannot do without
    exact(case, seed)   the same outputs from plain torch, in 64 bits
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "accelerating-tc_amd"))

import tcamd  # noqa: E402
from tcamd import batch as tbatch  # noqa: E402
from tcamd import learned as tlearned  # noqa: E402

ORIENT = {"degree": tcamd.ORIENT_DEGREE, "adir": tcamd.ORIENT_ADIR,
          "degeneracy": tcamd.ORIENT_DEGENERACY}
METHODS = ("hu", "bisson", "fox", "tricore")
WEDGES_MAX = 4_000_000_000  # exact() gives up beyond this many two-paths


def listed():
    return [
        # The benchmark's smallest graph, counted again and again while it
        # stays in device memory: launches and latency.
        dict(name="er65k-auto", do="count", graph="er", n=65536, records=1048576,
             orient="adir", engine="auto"),
        # One small edge list from host records to the count and back, as a
        # service that gets many small graphs one by one does it.
        dict(name="er3k-oneshot", do="oneshot", graph="er", n=3001, records=20011,
             orient="degree"),
        # The reference programs' whole run on a mid-sized skewed graph:
        # upload, degree orientation, CSR, schedule, count.
        dict(name="rmat18-oneshot", do="oneshot", graph="rmat", scale=18, records=4194304,
             orient="degree"),
        # The same with the A-direction peel, on a large graph.
        dict(name="rmat21-adir-oneshot", do="oneshot", graph="rmat", scale=21, records=33554432,
             orient="adir"),
        # The headline engine (shipped cost model) and preparation (A-order,
        # A-direction) on a large skewed graph that stays in device memory.
        dict(name="rmat23-learned", do="count", graph="rmat", scale=23, records=134217728,
             aorder=True, orient="adir", engine="learned"),
        # A scale-free graph of short lists: every task fits one lane.
        dict(name="ba3m-auto", do="count", graph="ba", n=3000017, k=8, orient="adir",
             engine="auto"),
        # Many small graphs counted by one replay (the batched workload).
        dict(name="batch384", do="batch", graphs=384, n_min=64, n_max=65536),
        # 4-cliques of a spatial graph: narrow roots.
        dict(name="rgg250k-k4", do="kclique", graph="rgg", n=250007, deg=48, k=4),
        # 5-cliques of a skewed graph: wide roots, deep trees.
        dict(name="rmat16-k5", do="kclique", graph="rmat", scale=16, records=2097152, k=5),
        # Triangles per vertex (clustering coefficients, feature extraction).
        dict(name="rmat20-vertex", do="vertex", graph="rmat", scale=20, records=16777216,
             orient="degree"),
        # The reference's own methods, for users who compare or switch.
        dict(name="rmat19-hu", do="count", graph="rmat", scale=19, records=8388608,
             orient="degree", engine="hu"),
        dict(name="rmat19-tricore", do="count", graph="rmat", scale=19, records=8388608,
             orient="adir", engine="tricore"),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, most):
    """A graph of up to `most` records."""
    kind = rng.choice(["er", "rmat", "rmat", "ba", "rgg"])
    m = _log(rng, 20_000, most)
    deg = _log(rng, 8, 64)  # records per vertex, both ends counted
    if kind == "rmat":
        return dict(graph="rmat", scale=max(8, int(round(math.log2(2 * m / deg)))), records=m)
    if kind == "ba":
        k = rng.randint(4, 16)
        return dict(graph="ba", n=max(100, min(m, 20_000_000) // k), k=k)
    if kind == "rgg":
        return dict(graph="rgg", n=max(500, min(m, 8_000_000) // 24), deg=rng.randint(16, 64))
    n = max(200, 2 * m // deg)
    return dict(graph="er", n=n, records=min(m, n * (n - 1) // 4))


def draw(rng):
    do = rng.choice(["count", "count", "oneshot", "oneshot", "method", "batch", "kclique",
                     "vertex"])
    if do == "count":
        c = dict(do="count", engine=rng.choice(["auto", "learned"]),
                 orient=rng.choice(["degree", "adir"]), **_draw_graph(rng, 60_000_000))
        if c["graph"] == "rmat":  # with and without the relabelling of the headline case
            c["aorder"] = rng.random() < 0.5
        return c
    if do == "oneshot":
        return dict(do="oneshot", orient=rng.choice(["degree", "adir"]),
                    **_draw_graph(rng, 30_000_000))
    if do == "method":
        return dict(do="count", engine=rng.choice(METHODS), orient=rng.choice(["degree", "adir"]),
                    **_draw_graph(rng, 8_000_000))
    if do == "batch":
        return dict(do="batch", graphs=_log(rng, 16, 384), n_min=64, n_max=_log(rng, 2000, 65536))
    if do == "kclique":
        if rng.random() < 0.5:
            return dict(do="kclique", graph="rgg", n=_log(rng, 2000, 250_000),
                        deg=rng.randint(24, 48), k=rng.choice([3, 4, 5]))
        scale = rng.randint(12, 16)
        return dict(do="kclique", graph="rmat", scale=scale, records=_log(rng, 8, 30) << scale,
                    k=rng.choice([3, 4, 5]))
    return dict(do="vertex", orient=rng.choice(["degree", "adir"]),
                **_draw_graph(rng, 16_000_000))


def _records(case, seed):
    kind = case["graph"]
    if kind == "rmat":
        return tcamd.gen_rmat(case["scale"], case["records"], 0.57, 0.19, 0.19, seed + 1)
    if kind == "er":
        return tcamd.gen_er(case["n"], case["records"], seed + 1)
    if kind == "ba":
        return tcamd.gen_ba(case["n"], case["k"], seed + 1)
    return tcamd.gen_rgg(case["n"], tcamd.rgg_radius(case["n"], case["deg"]), seed + 1)


def prepare(case, seed):
    ctx = tcamd.Context(0)
    state = {"case": case, "ctx": ctx}
    if case["do"] == "batch":
        state["batch"] = ctx.batch(tbatch.make_batch(case["graphs"], seed + 1,
                                                     n_min=case["n_min"], n_max=case["n_max"]))
        return state
    src, dst = _records(case, seed)
    if case["do"] == "oneshot":  # host records: the call takes them all the way
        state["src"], state["dst"] = src, dst
        return state
    # the per-vertex result has an entry for every vertex, isolated ones too
    g = ctx.graph(src, dst, _sizes(case)[0] if case["do"] == "vertex" else 0)
    if case.get("aorder"):
        g.relabel_aorder()
    g.orient(ORIENT["degeneracy" if case["do"] == "kclique" else case["orient"]])
    state["graph"] = g
    if case.get("engine") == "learned":
        state["model"] = tlearned.load(ctx)
    return state


def run(state):
    case = state["case"]
    if case["do"] == "batch":
        counts, _ = state["batch"].count()
        return {"counts": counts.astype(np.int64)}
    if case["do"] == "oneshot":
        g = state["ctx"].graph(state["src"], state["dst"])
        g.orient(ORIENT[case["orient"]])
        count = g.count().count
        i = g.info()
        g.close()
        return {"count": count, "edges": i.m_oriented, "max_out": i.max_out_degree,
                "sum_out_sq": i.sum_out_sq, "sum_in_out": i.sum_in_out}
    g = state["graph"]
    if case["do"] == "kclique":
        return {"count": g.kclique(case["k"]).count}
    if case["do"] == "vertex":
        return {"triangles": g.count_per_vertex().astype(np.int64)}
    if case["engine"] == "learned":
        return {"count": g.count_learned(state["model"]).count}
    return {"count": g.count(case["engine"]).count}


def _sizes(case):
    """(vertices, records) of a case, from its fields."""
    if case["do"] == "batch":
        mean_n = (case["n_max"] - case["n_min"]) / math.log(case["n_max"] / case["n_min"])
        return int(case["graphs"] * mean_n), int(case["graphs"] * mean_n * 17)
    kind = case["graph"]
    if kind == "rmat":
        return 1 << case["scale"], case["records"]
    if kind == "ba":
        return case["n"], case["n"] * case["k"]
    if kind == "rgg":
        return case["n"], case["n"] * case["deg"] // 2
    return case["n"], case["records"]


def work(case):
    n, m = _sizes(case)
    if case["do"] == "oneshot":
        return {"bytes": 8.0 * m + 48, "flops": 0.0}  # the records in, five numbers out
    out = {"vertex": 8.0 * n, "batch": 8.0 * case.get("graphs", 0)}.get(case["do"], 8.0)
    return {"bytes": 4.0 * (n + 1) + 4.0 * m + out, "flops": 0.0}  # the oriented CSR in


def _forward(src, dst, n, per_vertex):
    """Degree-oriented CSR sizes and forward counts of one graph by closing
    every two-path u -> v -> w, in int64; None beyond WEDGES_MAX two-paths."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    s = torch.from_numpy(np.asarray(src).astype(np.int64)).to(dev)
    d = torch.from_numpy(np.asarray(dst).astype(np.int64)).to(dev)
    deg = torch.bincount(s, minlength=n) + torch.bincount(d, minlength=n)
    swap = (deg[s] > deg[d]) | ((deg[s] == deg[d]) & (s < d))
    u, v = torch.where(swap, d, s), torch.where(swap, s, d)
    key = torch.unique((u * n + v)[u != v])
    u, v = key // n, key % n
    out = torch.bincount(u, minlength=n)
    start = torch.cumsum(out, 0) - out
    ind = torch.bincount(v, minlength=n)
    res = {"edges": int(key.numel()), "max_out": int(out.max()) if n else 0,
           "sum_out_sq": int((out * out).sum()), "sum_in_out": int((out * ind).sum())}
    if res["sum_in_out"] > WEDGES_MAX:
        return None
    tri = torch.zeros(n if per_vertex else 1, dtype=torch.int64, device=dev)
    lens = out[v]
    ends = torch.cumsum(lens, 0)
    lo = 0
    while lo < key.numel():
        base = int(ends[lo - 1]) if lo else 0
        hi = int(torch.searchsorted(ends, torch.tensor(base + 40_000_000, device=dev)))
        hi = min(max(hi, lo + 1), key.numel())
        ln = lens[lo:hi]
        e = torch.repeat_interleave(torch.arange(lo, hi, device=dev), ln)
        at = torch.arange(e.numel(), device=dev) - (ends[e] - lens[e] - base)
        w = v[start[v[e]] + at]
        want = u[e] * n + w
        pos = torch.searchsorted(key, want).clamp_(max=key.numel() - 1)
        hit = (key[pos] == want).to(torch.int64)
        if per_vertex:
            tri.index_add_(0, u[e], hit)
        else:
            tri += hit.sum()
        lo = hi
    res["tri"] = tri.cpu().numpy()
    return res


def exact(case, seed):
    if case["do"] == "kclique":
        return None
    if case["do"] == "batch":
        if case["graphs"] > 48:
            return None
        c = [int(_forward(s, d, n, False)["tri"][0]) if len(s) else 0
             for s, d, n in tbatch.make_batch(case["graphs"], seed + 1, n_min=case["n_min"],
                                              n_max=case["n_max"])]
        return {"counts": np.array(c, np.int64)}
    if _sizes(case)[1] > 40_000_000 or (case["do"] == "vertex" and case["orient"] != "degree"):
        return None
    src, dst = _records(case, seed)
    n = _sizes(case)[0] if case["do"] == "vertex" else int(max(src.max(), dst.max())) + 1
    r = _forward(src, dst, n, case["do"] == "vertex")
    if r is None:
        return None
    if case["do"] == "vertex":
        return {"triangles": r["tri"]}
    if case["do"] == "count":
        return {"count": int(r["tri"][0])}
    sizes = ("max_out", "sum_out_sq", "sum_in_out")  # the A-direction DAG has its own
    return {"count": int(r["tri"][0]), "edges": r["edges"],
            **{k: r[k] if case["orient"] == "degree" else None for k in sizes}}
