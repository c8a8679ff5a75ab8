"""The work users have this framework do, as measurable cases.

Every case goes through a public entry point: the Python facade (``EmbeddingPropagator``,
``NodeEmbedder``) or the C ABI of include/cloverleaf_ep.h through its ctypes binding
(``_native.Context`` / ``_native.Aligner``), which a program uses when it keeps the graph
resident on the GPU.

op     what a pass is
fit    EmbeddingPropagator.learn_features: the whole call, from host arrays to a table
learn  a resident context: draw the initial table, train `passes` passes, read the table
step   ep_step_explicit_noalloc on explicit samples, then the updated table (serving loop)
embed  NodeEmbedder.embed_feature_set: host feature lists and table in, node rows out
align  NeighborhoodAligner on a resident graph: one run over a range of nodes

Sizes are those of the named workloads of cloverleaf_amd/synth.py and of the tests, with
the node count cut to what trains in well under two seconds; batch sizes, widths, sample
sizes and feature distributions are the workloads' own.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cloverleaf_amd import (EmbeddingPropagator, EPLoss, FeatureAggregator, FeatureSet, Graph, LossWeighting,
                            NodeEmbedder, NodeEmbeddings, Vocab)
from cloverleaf_amd import _native as N
from cloverleaf_amd import synth

COUNTS = {"poisson": synth.COUNT_POISSON, "uniform": synth.COUNT_UNIFORM, "loguniform": synth.COUNT_LOGUNIFORM}

# Fields of a training case and their defaults (the reference's, where it has one).
TRAIN = dict(nodes=2000, edges=10000, beta=2.5, dmax=100, directed=False, fkind="poisson", f1=7.0, f2=0.0, vocab=4000,
             zipf=1.1, dims=100, batch=50, negatives=1, max_nodes=0, passes=2, alpha=0.01, gamma=0.5, loss="margin",
             valid=0.1, precision="fp32", fp16_adjoints=False, concurrent=1, graph=False, exact_grad=False, log_weight=False,
             hard=0, weighted=False, max_features=0, heads=0, dk=0)


def _train(name, op, **kw):
    c = dict(TRAIN, op=op, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: an online update of 64 anchors with samples the program drew itself
        _train("step-64", "step", nodes=3000, edges=30000, vocab=1000, dims=64, batch=64, negatives=5, max_nodes=10),
        # the reference's defaults (d=100, batch 50, one negative, every neighbour, 10% held out) on a small graph
        _train("fit-defaults", "fit", alpha=0.9, gamma=1.0, passes=3),
        # the 10k-node workload: short steps, launches count
        _train("learn-10k", "learn", nodes=10_000, edges=100_000, dmax=1000, vocab=50_000, dims=64, batch=128, negatives=5,
               max_nodes=10, passes=5),
        # random-walk positives (PPR loss), exact gradients, a BF16 table, two batches a step: options in ordinary use
        _train("learn-ppr-bf16", "learn", nodes=30_000, edges=300_000, dmax=1000, vocab=30_000, dims=32, batch=512,
               negatives=8, max_nodes=10, passes=3, loss="ppr", precision="bf16", concurrent=2, exact_grad=True),
        # the 1M-node workload's shape, one batch per step in FP32
        _train("learn-1m-plain", "learn", nodes=100_000, edges=2_000_000, beta=2.2, dmax=10_000, fkind="uniform", f1=1.0,
               f2=32.0, vocab=100_000, dims=128, batch=1024, negatives=10, max_nodes=20, passes=3),
        # the same shape, eight batches per step replayed from a graph
        _train("learn-1m-batched", "learn", nodes=200_000, edges=4_000_000, beta=2.2, dmax=10_000, fkind="uniform", f1=1.0,
               f2=32.0, vocab=200_000, dims=128, batch=1024, negatives=10, max_nodes=20, passes=4, concurrent=8, graph=True,
               valid=0.0),
        # the 10M-node workload's shape: d=256, long ragged feature lists (1 to 128), directed graph
        _train("learn-10m", "learn", nodes=100_000, edges=2_000_000, beta=2.1, dmax=10_000, directed=True, fkind="loguniform",
               f1=1.0, f2=128.0, vocab=200_000, zipf=1.05, dims=256, batch=8192, negatives=20, max_nodes=32, passes=3,
               valid=0.0),
        # the 50M-node workload's shape, the largest: BF16 table, FP32 master, FP16 adjoint rows, 131072 anchors a step
        _train("learn-50m-bf16", "learn", nodes=300_000, edges=6_000_000, beta=2.2, dmax=10_000, fkind="uniform", f1=1.0,
               f2=64.0, vocab=120_000, dims=256, batch=16384, negatives=20, max_nodes=20, passes=6, concurrent=8,
               graph=True, precision="bf16-master", fp16_adjoints=True, valid=0.0),
        # the attention workload's shape: rows of 768 (4 heads, d_k 32, d 128), up to 64 features per node
        _train("learn-attention", "learn", nodes=20_000, edges=400_000, beta=2.3, dmax=2000, fkind="uniform", f1=1.0, f2=64.0,
               vocab=20_000, dims=128, batch=1024, negatives=10, max_nodes=20, passes=2, heads=4, dk=32, valid=0.0),
        # node embeddings from learned feature rows, after training: the plain mean
        dict(name="embed-averaged", op="embed", kind="averaged", nodes=100_000, fkind="uniform", f1=1.0, f2=32.0,
             vocab=50_000, zipf=1.1, dims=128, heads=0, dk=0),
        # the same through attention
        dict(name="embed-attention", op="embed", kind="attention", nodes=40_000, fkind="uniform", f1=1.0, f2=32.0,
             vocab=20_000, zipf=1.1, dims=128, heads=4, dk=32),
        # smoothing node embeddings over a resident graph
        dict(name="align-100k", op="align", nodes=100_000, edges=2_000_000, beta=2.2, dmax=10_000, dims=128, alpha=0.5,
             max_neighbors=0),
    ]


# ---------------------------------------------------------------------------------------
# draws
# ---------------------------------------------------------------------------------------
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mean_features(c):
    if c["fkind"] == "poisson":
        return 1.0 + c["f1"]
    if c["fkind"] == "uniform":
        return (c["f1"] + c["f2"]) / 2.0
    return (c["f2"] - c["f1"]) / math.log(c["f2"] / c["f1"])


def _occurrences(c):
    """Feature occurrences of one example, on average."""
    deg = c["edges"] * (1 if c["directed"] else 2) / c["nodes"]
    s = c["negatives"] if c["loss"] == "ppr" else (deg if c["max_nodes"] == 0 else min(c["max_nodes"], deg))
    f = _mean_features(c)
    return (1.0 + s + c["negatives"]) * (min(f, c["max_features"]) if c["max_features"] else f)


def _width(c):
    return c["heads"] * (2 * c["dk"] + c["dims"]) if c["heads"] else c["dims"]


def _draw_features(rng, c, most):
    k = rng.random()
    if k < 0.34:
        c.update(fkind="poisson", f1=float(rng.randint(1, 12)), f2=0.0)
    elif k < 0.8:
        c.update(fkind="uniform", f1=1.0, f2=float(_log(rng, 4, min(64, most))))
    else:
        c.update(fkind="loguniform", f1=1.0, f2=float(_log(rng, 8, most)))
    c.update(zipf=round(rng.uniform(1.02, 1.3), 3))


def _draw_train(rng):
    c = _train("", "learn")
    batch = _log(rng, 24, 8192)
    c.update(batch=batch, dims=rng.choice([8, 16, 32, 64, 100, 128, 128, 256, 256]), negatives=_log(rng, 1, 25),
             max_nodes=_log(rng, 3, 40), passes=rng.randint(1, 4), concurrent=rng.choice([1, 1, 1, 2, 4, 8]),
             graph=rng.random() < 0.4, beta=round(rng.uniform(2.05, 2.6), 2), directed=rng.random() < 0.25,
             valid=rng.choice([0.0, 0.1]), gamma=rng.choice([0.5, 1.0]), exact_grad=rng.random() < 0.2,
             log_weight=rng.random() < 0.15)
    c["nodes"] = max(400, min(150_000, int(batch * rng.uniform(2.5, 60.0))))
    c["edges"] = c["nodes"] * rng.randint(3, 20)
    c["dmax"] = max(20, c["nodes"] // 20)
    _draw_features(rng, c, 128)
    c["vocab"] = max(200, int(c["nodes"] * rng.uniform(0.3, 3.0)))
    p = rng.random()
    if p < 0.35:
        c.update(precision=rng.choice(["bf16", "bf16-master"]), fp16_adjoints=rng.random() < 0.6)
    k = rng.random()
    if k < 0.12:
        c.update(loss=rng.choice(["contrastive", "starspace", "rank", "rankspace", "ppr"]))
    elif k < 0.2:
        c.update(hard=rng.randint(1, c["negatives"]))
    elif k < 0.28:
        c.update(weighted=True)
    elif k < 0.34 and c["f2"] <= 64:
        c.update(max_features=rng.randint(2, 12))
    elif k < 0.46:
        c.update(heads=rng.choice([1, 2, 4]), dk=rng.choice([8, 16, 32]), dims=rng.choice([64, 128]), fp16_adjoints=False,
                 batch=min(c["batch"], 1024), concurrent=min(c["concurrent"], 2), max_nodes=min(c["max_nodes"], 20))
        c["f2"] = min(c["f2"], 64.0)
        # row widths the table kernels are built for
        if _width(c) not in (64, 100, 128, 256, 384, 512, 768):
            c.update(heads=4, dk=32, dims=128)
        c["nodes"] = min(c["nodes"], 20_000)
        c["edges"] = min(c["edges"], 15 * c["nodes"])
    return c


def _fmax(c):
    return 40 if c["fkind"] == "poisson" else int(c["f2"])


def _fits(c):
    """At most half of the largest listed case's work, the documented limits, bounded buffers."""
    top = 300_000 * 6 * 41 * 32.5 * 256
    if c["nodes"] * c["passes"] * _occurrences(c) * _width(c) * (6 if c["heads"] else 1) > top / 2:
        return False
    entries = 1 + (c["negatives"] if c["loss"] == "ppr" else c["max_nodes"]) + c["negatives"]
    keys = c["batch"] * c["concurrent"] * entries * _fmax(c)
    return entries * _fmax(c) <= 8000 and keys * (_width(c) * 4 if c["heads"] else 64 + _width(c) // 4) < 25e9


def draw(rng):
    k = rng.random()
    if k < 0.6:
        while True:
            c = _draw_train(rng)
            if _fits(c):
                return c
    if k < 0.7:  # whole calls at and around the defaults
        c = _train("", "fit", nodes=_log(rng, 300, 6000), dims=rng.choice([32, 64, 100, 100, 128]), batch=rng.choice([32, 50, 50, 128]),
                   negatives=rng.randint(1, 6), passes=rng.randint(1, 5), alpha=rng.choice([0.9, 0.1, 0.01]), gamma=1.0,
                   max_nodes=rng.choice([0, 0, 5, 10]))
        c.update(edges=c["nodes"] * rng.randint(3, 8), dmax=60, vocab=max(100, int(c["nodes"] * rng.uniform(0.5, 3.0))),
                 f1=float(rng.randint(1, 9)))
        return c
    if k < 0.8:
        return _train("", "step", nodes=_log(rng, 500, 20_000), edges=0, vocab=_log(rng, 300, 4000), dims=rng.choice([32, 64, 100, 128, 256]),
                      batch=_log(rng, 1, 200), negatives=rng.randint(1, 10), max_nodes=rng.randint(2, 12), f1=float(rng.randint(1, 9)))
    if k < 0.92:
        att = rng.random() < 0.4
        c = dict(op="embed", kind="attention" if att else "averaged", nodes=_log(rng, 500, 40_000 if att else 150_000),
                 vocab=_log(rng, 500, 60_000), dims=128 if att else rng.choice([8, 32, 64, 100, 128, 256]), heads=4 if att else 0,
                 dk=32 if att else 0)
        _draw_features(rng, c, 64)
        return c
    c = dict(op="align", nodes=_log(rng, 1000, 120_000), beta=round(rng.uniform(2.05, 2.6), 2), dims=rng.choice([32, 64, 100, 128, 256]),
             alpha=rng.choice([0.0, 0.3, 0.5, -1.0]), max_neighbors=rng.choice([0, 0, 10, 33]))
    c.update(edges=c["nodes"] * rng.randint(3, 20), dmax=max(20, c["nodes"] // 10))
    return c


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _graph(c, seed):
    return synth.chung_lu(c["nodes"], c["edges"], c["beta"], float(c["dmax"]), c.get("directed", False), 3 * seed + 1)


def _features(c, seed):
    return synth.features(c["nodes"], COUNTS[c["fkind"]], c["f1"], c["f2"], c["vocab"], c["zipf"], 3 * seed + 2)


def _row_cdf(indptr, seed):
    """Per-row CDF of random edge weights."""
    ip = indptr.astype(np.int64)
    w = np.random.default_rng(seed).uniform(0.1, 1.0, size=int(ip[-1]))
    tot = np.concatenate([[0.0], np.cumsum(w)])
    deg = np.diff(ip)
    start, end = np.repeat(tot[ip[:-1]], deg), np.repeat(tot[ip[1:]], deg)
    cdf = ((tot[1:] - start) / np.maximum(end - start, 1e-300)).astype(np.float32)
    cdf[ip[1:][deg > 0] - 1] = 1.0
    return np.minimum(cdf, np.float32(1.0))


def _config(c, seed):
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.passes = c["dims"], c["batch"], c["negatives"], c["passes"]
    cfg.alpha, cfg.gamma, cfg.valid_pct, cfg.seed = c["alpha"], c["gamma"], c["valid"], 20222022 + seed
    if c["max_nodes"]:
        cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, c["max_nodes"]
    cfg.loss_kind = N.LOSS_KINDS[c["loss"]]
    cfg.loss_param2 = 0.25 if c["loss"] in ("ppr", "contrastive") else 0.0
    cfg.precision = {"fp32": N.EP_PREC_FP32, "bf16": N.EP_PREC_BF16, "bf16-master": N.EP_PREC_BF16_MASTER}[c["precision"]]
    cfg.fp16_adjoints, cfg.concurrent_batches = int(c["fp16_adjoints"]), c["concurrent"]
    cfg.use_graph, cfg.grad_mode = int(c["graph"]), N.EP_GRAD_EXACT if c["exact_grad"] else N.EP_GRAD_FIRST_LEAF
    cfg.loss_weighting = N.EP_LW_LOG if c["log_weight"] else N.EP_LW_NONE
    cfg.hard_negatives = c["hard"]
    if c["weighted"]:
        cfg.weighted_neighbor_sampling = cfg.weighted_neighbor_averaging = 1
    if c["max_features"]:
        cfg.max_features_kind, cfg.max_features = N.EP_SAMPLE_FIXED, c["max_features"]
    if c["heads"]:
        cfg.attention_heads, cfg.attention_dk = c["heads"], c["dk"]
    return cfg


def _unit_rows(vocab, width, seed):
    x = torch.rand((vocab, width), generator=torch.Generator("cuda").manual_seed(seed), device="cuda") * 2.0 - 1.0
    return (x / x.norm(dim=1, keepdim=True)).cpu().numpy()


def _step_inputs(c, seed):
    """Explicit samples of one step: anchors, neighbour counts and lists, negatives."""
    rng = np.random.default_rng(seed)
    f_indptr, f_ids = _features(c, seed)
    b, s, k = c["batch"], c["max_nodes"], c["negatives"]
    anchors = rng.choice(c["nodes"], size=b, replace=False).astype(np.uint32)
    cnt = rng.integers(1, s + 1, size=b).astype(np.uint32)
    nbr = rng.integers(0, c["nodes"], size=(b, s)).astype(np.uint32)
    neg = rng.integers(0, c["nodes"], size=(b, k)).astype(np.uint32)
    return f_indptr, f_ids, _unit_rows(c["vocab"], c["dims"], seed), anchors, cnt, nbr, neg


def prepare(case, seed):
    c = case
    if c["op"] == "fit":
        indptr, indices = _graph(c, seed)
        g = Graph.from_csr(indptr, indices)
        fs = FeatureSet.from_csr(g, *_features(c, seed), c["vocab"])
        ep = EmbeddingPropagator(alpha=c["alpha"], loss=EPLoss.margin(c["gamma"], c["negatives"]), batch_size=c["batch"],
                                 dims=c["dims"], passes=c["passes"], seed=20222022 + seed, max_nodes=c["max_nodes"] or None,
                                 valid_pct=c["valid"], loss_weighting=LossWeighting.Log() if c["log_weight"] else None,
                                 indicator=False, precision=c["precision"], concurrent_batches=c["concurrent"])
        return {"op": "fit", "ep": ep, "graph": g, "features": fs}
    if c["op"] == "learn":
        ctx = N.Context(_config(c, seed))
        indptr, indices = _graph(c, seed)
        ctx.set_graph(indptr, indices)
        if c["weighted"]:
            ctx.set_edge_weights(_row_cdf(indptr, seed))
        ctx.set_features(*_features(c, seed), c["vocab"])
        return {"op": "learn", "ctx": ctx}
    if c["op"] == "step":
        f_indptr, f_ids, table, anchors, cnt, nbr, neg = _step_inputs(c, seed)
        ctx = N.Context(_config(c, seed))
        ctx.set_graph(np.arange(c["nodes"] + 1, dtype=np.uint64), np.arange(c["nodes"], dtype=np.uint32))
        ctx.set_features(f_indptr, f_ids, c["vocab"])
        ctx.set_table(table)
        return {"op": "step", "ctx": ctx, "args": (anchors, cnt, nbr, neg), "lr": c["alpha"]}
    if c["op"] == "embed":
        vocab = Vocab.anonymous(c["nodes"])
        g = Graph(np.zeros(c["nodes"] + 1, dtype=np.uint64), np.zeros(0, dtype=np.uint32), None, vocab)
        fs = FeatureSet.from_csr(g, *_features(c, seed), c["vocab"])
        agg = FeatureAggregator.Attention(c["heads"], c["dk"]) if c["kind"] == "attention" else FeatureAggregator.Averaged()
        emb = NodeEmbeddings(fs.feature_vocab, _unit_rows(c["vocab"], _width(c), seed))
        return {"op": "embed", "embedder": NodeEmbedder(agg), "features": fs, "table": emb}
    indptr, indices = _graph(c, seed)
    emb = _unit_rows(c["nodes"], c["dims"], seed)
    return {"op": "align", "aligner": N.Aligner(indptr, indices, _row_cdf(indptr, seed), emb),
            "alpha": None if c["alpha"] < 0 else c["alpha"], "max_neighbors": c["max_neighbors"] or None}


def run(state):
    op = state["op"]
    if op == "fit":
        out = state["ep"].learn_features(state["graph"], state["features"])
        return {"table": out.embeddings, "train": [h["train"] for h in state["ep"].history],
                "valid": [h["valid"] for h in state["ep"].history]}
    if op == "learn":
        losses = []
        ctx = state["ctx"]
        ctx.set_table(None)
        ctx.learn(lambda p, step, train, valid, lr: losses.append(train))
        return {"table": ctx.get_table(), "train": losses}
    if op == "step":
        loss = state["ctx"].step_explicit_noalloc(*state["args"], 1, state["lr"])
        return {"loss": loss, "table": state["ctx"].get_table()}
    if op == "embed":
        return state["embedder"].embed_feature_set(state["features"], state["table"]).embeddings
    return state["aligner"].run(state["alpha"], state["max_neighbors"])


# ---------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------
def _distinct(occurrences, vocab, zipf):
    """Expected distinct features among `occurrences` Zipf draws."""
    p = np.arange(1, vocab + 1, dtype=np.float64) ** -zipf
    return float(-np.expm1(occurrences * np.log1p(-p / p.sum())).sum())


def work(case):
    c = case
    if c["op"] == "align":
        e = c["edges"] * 2.0
        if c["max_neighbors"]:
            e = min(e, float(c["nodes"]) * c["max_neighbors"])
        d = c["dims"]
        return {"bytes": c["nodes"] * (2.0 * d * 4 + 8) + 8 * e, "flops": 2 * e * d + 3.0 * c["nodes"] * d}
    f = _mean_features(c)
    w = _width(c)
    if c["op"] == "embed":
        occ = c["nodes"] * f
        flops = occ * w
        if c["kind"] == "attention":  # scores, softmax, weighted values
            flops = c["nodes"] * c["heads"] * (2 * c["dk"] * f * f + f * f + 2 * c["dims"] * f)
        return {"bytes": 4.0 * c["vocab"] * w + 4 * occ + 8 * c["nodes"] + 4.0 * c["nodes"] * c["dims"], "flops": flops}
    # a training step reads its distinct rows once and updates them (table row, both Adam
    # moments, the master where there is one); the ids of its occurrences are read once
    anchors = c["batch"] * c["concurrent"]
    train = c["nodes"] * (1.0 - c["valid"])
    steps = 1.0 if c["op"] == "step" else c["passes"] * max(1.0, train / anchors)
    occ = _occurrences(c) if c["op"] != "step" else (1 + (c["max_nodes"] + 1) / 2 + c["negatives"]) * f
    per_step = min(anchors, c["nodes"]) * occ
    rows = _distinct(per_step, c["vocab"], c["zipf"])
    b = 4 if c["precision"] == "fp32" else 2
    value = 16 + 2 * b if c["precision"] != "bf16-master" else 24 + 2 * b
    flops = steps * (3 * per_step * w + 12 * rows * w)
    if c["heads"]:
        blocks = min(anchors, c["nodes"]) * occ / f
        flops = steps * 3 * blocks * c["heads"] * (2 * c["dk"] * f * f + f * f + 2 * c["dims"] * f)
    table = 0.0 if c["op"] == "step" else 4.0 * c["vocab"] * w  # the initial table written
    return {"bytes": steps * (rows * w * value + 4 * per_step) + table + 4.0 * c["vocab"] * w, "flops": flops}


# ---------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------
def _exact_step(c, seed):
    """Margin loss, first-leaf gradients, one lazy Adam update: float64 numpy."""
    f_indptr, f_ids, table, anchors, cnt, nbr, neg = _step_inputs(c, seed)
    t = table.astype(np.float64)
    ip = f_indptr.astype(np.int64)

    def occurrences(nodes):
        return np.concatenate([f_ids[ip[u]:ip[u + 1]] for u in nodes]).astype(np.int64)

    grads, losses = {}, np.zeros(len(anchors))
    for i, v in enumerate(anchors):
        cons = [occurrences([v]), occurrences(nbr[i, :cnt[i]])] + [occurrences([u]) for u in neg[i]]
        x = [t[o].mean(axis=0) for o in cons]
        a, p = x[0], x[1]
        dist = [np.linalg.norm(p - y) for y in [a] + x[2:]]
        terms = [c["gamma"] + dist[0] - d for d in dist[1:]]
        on = [l > 0 for l in terms]
        if not any(on):
            continue
        losses[i] = sum(l for l, k in zip(terms, on) if k) / sum(on)
        gp = (p - a) / dist[0]
        adj = [-gp, gp]
        for y, d, k in zip(x[2:], dist[1:], on):
            g = (p - y) / d / sum(on) if k else None
            adj.append(g)
            if k:
                adj[1] = adj[1] - g
        seen = set()
        for o, g in zip(cons, adj):
            if g is None or not np.isfinite(g).all():
                continue
            ids, mult = np.unique(o, return_counts=True)
            for f, m in zip(ids.tolist(), mult.tolist()):
                if f not in seen:
                    seen.add(f)
                    grads[f] = grads.get(f, 0.0) + g * (m / len(o))
    for f, g in grads.items():
        m, v2 = 0.1 * g / (1 - 0.9 ** 2), 0.001 * g * g / (1 - 0.999 ** 2)
        t[f] -= c["alpha"] * m / (np.sqrt(v2) + 1e-8)
    return {"loss": losses, "table": t}


def _segments(indptr):
    ip = torch.from_numpy(indptr.astype(np.int64))
    return torch.repeat_interleave(torch.arange(len(ip) - 1), ip[1:] - ip[:-1]), ip[1:] - ip[:-1]


def exact(case, seed):
    c = case
    if c["op"] == "step":
        return _exact_step(c, seed)
    if c["op"] == "align":
        indptr, indices = _graph(c, seed)
        cdf = torch.from_numpy(_row_cdf(indptr, seed)).double()
        emb = torch.from_numpy(_unit_rows(c["nodes"], c["dims"], seed)).double().cuda()
        seg, deg = _segments(indptr)
        first = torch.from_numpy(indptr.astype(np.int64))[:-1][seg]
        pos = torch.arange(len(seg)) - first
        p = torch.where(pos == 0, cdf, cdf - torch.roll(cdf, 1))
        if c["max_neighbors"]:
            p = torch.where(pos < c["max_neighbors"], p, torch.zeros_like(p))
        out = torch.zeros_like(emb)
        ids, seg, p = torch.from_numpy(indices.astype(np.int64)).cuda(), seg.cuda(), p.cuda()
        for s in range(0, len(ids), 1 << 20):
            k = slice(s, s + (1 << 20))
            out.index_add_(0, seg[k], emb[ids[k]] * p[k, None])
        if c["alpha"] < 0:
            a = torch.clamp(1.0 / torch.log(deg.double() + 1.0), max=1.0).cuda()[:, None]
        else:
            a = float(np.float32(c["alpha"]))
        return ((1 - a) * out + a * emb).cpu().numpy()
    if c["op"] == "embed":
        f_indptr, f_ids = _features(c, seed)
        table = torch.from_numpy(_unit_rows(c["vocab"], _width(c), seed)).double().cuda()
        if c["kind"] == "averaged":
            seg, n = _segments(f_indptr)
            ids, seg = torch.from_numpy(f_ids.astype(np.int64)).cuda(), seg.cuda()
            out = torch.zeros((c["nodes"], c["dims"]), dtype=torch.float64, device="cuda")
            for s in range(0, len(ids), 1 << 20):
                k = slice(s, s + (1 << 20))
                out.index_add_(0, seg[k], table[ids[k]])
            return (out / n.cuda()[:, None]).cpu().numpy()
        # Full attention over each node's listed features, one group per list length
        h, dk, dm = c["heads"], c["dk"], c["dims"]
        ip = torch.from_numpy(f_indptr.astype(np.int64))
        ids = torch.from_numpy(f_ids.astype(np.int64))
        n = ip[1:] - ip[:-1]
        out = torch.zeros((c["nodes"], dm), dtype=torch.float64)
        for length in torch.unique(n).tolist():
            for nodes in torch.split(torch.nonzero(n == length)[:, 0], 2000):
                rows = table[ids[ip[nodes][:, None] + torch.arange(length)].cuda()]
                v = rows[..., 2 * h * dk:].reshape(-1, length, h, dm)
                if length == 1:
                    out[nodes] = v[:, 0, 0].cpu()
                    continue
                q = rows[..., :h * dk].reshape(-1, length, h, dk).permute(0, 2, 1, 3).contiguous()
                k = rows[..., h * dk:2 * h * dk].reshape(-1, length, h, dk).permute(0, 2, 3, 1).contiguous()
                w = torch.softmax(torch.matmul(q, k) / math.sqrt(dk), dim=-1).sum(dim=2)
                out[nodes] = ((w.permute(0, 2, 1)[..., None] * v).sum(dim=(1, 2)) / (length * h)).cpu()
        return out.numpy()
    return None  # many steps of sampled training: no 64-bit trajectory stays near it
