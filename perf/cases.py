"""Performance cases of the label-propagation update, through the package's public calls.

Each case is one thing a program does with this library: hand over a graph and
run label propagation on it.  What a program keeps between runs -- the
context, the uploaded graph, the trained network -- is made in prepare();
run() is the call it then repeats.  Graphs come from the package's seeded
generators (planted partitions, R-MAT, LFR-style), with the parameters its
tests and benchmark use.

flow:
  run      Graph.run(iters): the whole label-propagation run, labels on the host
  steps    init, then step by step until the stop rule, as a program that
           watches the change counts does (and the command line's verbose run)
  learned  run() under learned dispatch with a network trained beforehand
  batch    run() over a batch of independent graphs, the loop captured
  ooc      run() with the neighbour array in host memory, streamed (policy 2)
  oneshot  upload, run, read the labels, free: what the command line does per file
  train    mlp_train: the training that learned dispatch needs once per graph
"""
import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np

from galp_amd import _abi

HIDDEN = 32          # the dispatcher's network: 4-32-32-1
CAND_THRESH = 14.0   # predicted distinct labels that take the candidate path
METHOD = {"hash": _abi.METHOD_HASH, "sort": _abi.METHOD_SORT}


def listed():
    return [
        # the smallest graphs of a batch when they are run one at a time: all launches and latency
        {"name": "hash-pp-1k", "flow": "run", "method": "hash", "family": "pp", "n": 1000, "community": 50,
         "intra": 8, "inter": 2, "iters": 10},
        # the small planted partition that both methods are compared on
        {"name": "hash-pp-16k", "flow": "run", "method": "hash", "family": "pp", "n": 16384, "community": 256,
         "intra": 8, "inter": 2, "iters": 10},
        {"name": "sort-pp-16k", "flow": "run", "method": "sort", "family": "pp", "n": 16384, "community": 256,
         "intra": 8, "inter": 2, "iters": 10},
        # a program that watches convergence, on a mid-sized skewed graph
        {"name": "steps-rmat-18", "flow": "steps", "method": "hash", "family": "rmat", "scale": 18, "ef": 16,
         "iters": 10},
        # the sort method on a mid-sized skewed graph with hub rows
        {"name": "sort-rmat-20", "flow": "run", "method": "sort", "family": "rmat", "scale": 20, "ef": 16,
         "iters": 10},
        # the in-core single-GPU configuration
        {"name": "hash-rmat-22", "flow": "run", "method": "hash", "family": "rmat", "scale": 22, "ef": 16,
         "iters": 10},
        # the largest in-core graph here: hubs of hundreds of tiles
        {"name": "hash-rmat-23", "flow": "run", "method": "hash", "family": "rmat", "scale": 23, "ef": 16,
         "iters": 10},
        # learned dispatch on the social-network-like graph it was made for, an odd number of vertices
        {"name": "learned-lfr-1m", "flow": "learned", "method": "hash", "family": "lfr", "n": 1000003,
         "avg_deg": 20.0, "max_deg": 2000, "mu": 0.3, "iters": 10},
        # many uneven graphs in one run
        {"name": "batch-512", "flow": "batch", "method": "hash", "family": "batch", "graphs": 512, "nmax": 20000,
         "iters": 10},
        # a graph whose neighbour array does not stay on the card
        {"name": "ooc-rmat-20", "flow": "ooc", "method": "hash", "family": "rmat", "scale": 20, "ef": 16,
         "buffer_pow": 22, "iters": 10},
        # the command line's job on one file: upload, run, labels
        {"name": "oneshot-lfr-300k", "flow": "oneshot", "method": "hash", "family": "lfr", "n": 300007,
         "avg_deg": 20.0, "max_deg": 2000, "mu": 0.3, "iters": 10},
        # the network's training on one graph's logged samples
        {"name": "train-100k", "flow": "train", "samples": 100003, "epochs": 8, "batch": 512},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: graphs of 1 thousand to 8 million vertices."""
    flow = rng.choice(["run", "run", "run", "run", "steps", "learned", "batch", "ooc", "oneshot", "train"])
    if flow == "train":
        return {"flow": "train", "samples": _log_uniform(rng, 5000, 50000), "epochs": rng.randint(2, 8),
                "batch": rng.randint(128, 512)}
    if flow == "batch":
        return {"flow": "batch", "method": "hash", "family": "batch", "graphs": _log_uniform(rng, 16, 512),
                "nmax": _log_uniform(rng, 2000, 20000), "iters": 10}
    case = {"flow": flow, "method": "hash" if flow in ("learned", "ooc") else rng.choice(["hash", "hash", "sort"])}
    case["family"] = rng.choice(["rmat", "lfr"] if flow in ("learned", "ooc") else ["pp", "rmat", "lfr"])
    if case["family"] == "pp":
        case.update(n=_log_uniform(rng, 1000, 1000000), community=rng.randint(32, 1024), intra=rng.randint(4, 24),
                    inter=rng.randint(1, 6))
    elif case["family"] == "rmat":
        top = {"run": 22, "steps": 21}.get(flow, 20)
        case.update(scale=rng.randint(13, top), ef=rng.randint(8, 16))
    else:
        case.update(n=_log_uniform(rng, 10000, 2000000 if flow == "run" else 1000000),
                    avg_deg=round(rng.uniform(10.0, 30.0), 2), max_deg=rng.randint(500, 2000),
                    mu=round(rng.uniform(0.1, 0.4), 3))
    if flow == "ooc":
        case["buffer_pow"] = rng.randint(18, 24)
    case["iters"] = 10
    return case


def _graph(case, seed):
    if case["family"] == "pp":
        return _abi.gen_planted_partition(case["n"], case["community"], case["intra"], case["inter"], seed)
    if case["family"] == "rmat":
        return _abi.gen_rmat(case["scale"], case["ef"], seed=seed)
    return _abi.gen_lfr(case["n"], avg_deg=case["avg_deg"], max_deg=case["max_deg"], mu=case["mu"], seed=seed)


def _batch(case, seed):
    """The batched configuration's graphs as one disjoint union: n ~ U[1000,
    nmax], community size ~ U[32, 1024], intra degree d ~ U[8, 48], inter
    degree d / 4.  The sizes belong to the case, the edges to the seed."""
    rng = np.random.default_rng(4096)
    spec = []
    for _ in range(case["graphs"]):
        d = int(rng.integers(8, 49))
        spec.append((int(rng.integers(1000, case["nmax"] + 1)), int(rng.integers(32, 1025)), (d + 1) // 2,
                     max(1, (d + 4) // 8)))
    with ThreadPoolExecutor(min(16, len(os.sched_getaffinity(0)))) as pool:
        parts = list(pool.map(lambda k: _abi.gen_planted_partition(*spec[k], seed * 100003 + k), range(len(spec))))
    vbase = np.concatenate([[0], np.cumsum([p[0] for p in spec])]).astype(np.int64)
    ebase = np.concatenate([[0], np.cumsum([len(nbr) for _, nbr in parts])]).astype(np.int64)
    off = np.empty(vbase[-1] + 1, np.int64)
    nbr = np.empty(ebase[-1], np.int32)
    for k, (o, u) in enumerate(parts):
        off[vbase[k]:vbase[k + 1]] = o[:-1] + ebase[k]
        nbr[ebase[k]:ebase[k + 1]] = u + np.int32(vbase[k])
    off[-1] = ebase[-1]
    return off, nbr, vbase


def _samples(count, seed):
    """Training samples of the kind a run logs: log2 of degree, neighbour
    degrees, the previous distinct count (-1 before the first), target log2
    of the distinct count."""
    rng = np.random.default_rng(seed)
    x = np.empty((count, 4), np.float32)
    x[:, 0] = rng.uniform(6, 16, count)
    x[:, 1] = rng.uniform(4, 12, count)
    x[:, 2] = x[:, 1] + rng.uniform(0, 8, count)
    x[:, 3] = np.where(rng.random(count) < 0.1, -1.0, x[:, 0] * rng.uniform(0.1, 1.0, count))
    y = np.where(x[:, 3] >= 0, 0.8 * x[:, 3] + 0.1 * x[:, 0], 0.9 * x[:, 0] - 0.2 * x[:, 1])
    return x, (y + rng.normal(0.0, 0.1, count)).astype(np.float32)


class State:
    """A program's context and graph, freed with the state."""

    def __init__(self, case):
        self.case, self.graph, self.ctx = case, None, _abi.Context(0)

    def __del__(self):
        if self.graph is not None:
            self.graph.free()
        self.ctx.close()


def prepare(case, seed):
    s = State(case)
    flow = case["flow"]
    if flow == "train":
        s.x, s.y = _samples(case["samples"], seed)
        s.params = _abi.mlp_init(HIDDEN, seed + 1)
        return s
    if flow == "batch":
        off, nbr, vbase = _batch(case, seed)
        s.graph = _abi.Graph(s.ctx, off, nbr, reorder=0, graph_capture=1)
        s.graph.set_batch(vbase)
        return s
    off, nbr = _graph(case, seed)
    method = METHOD[case["method"]]
    if flow == "oneshot":
        s.off, s.nbr = off, nbr
    elif flow == "ooc":
        s.graph = _abi.Graph(s.ctx, off, nbr, method=method, policy=_abi.POLICY_OOC_ASYNC,
                             buffer_pow=case["buffer_pow"])
    elif flow == "learned":
        with _abi.Graph(s.ctx, off, nbr) as g:
            g.log_enable((case["iters"] + 1) * max(int((np.diff(off) > 64).sum()), 1))
            g.run(case["iters"], want_labels=False)
            x, y = g.log_read()
        order = np.lexsort((y, x[:, 3], x[:, 2], x[:, 1], x[:, 0]))
        pick = order[np.random.default_rng(seed).choice(len(order), min(len(order), 40000), replace=False)]
        params = _abi.mlp_init(HIDDEN, 1)
        if len(pick):
            params, _ = _abi.mlp_train(s.ctx, HIDDEN, params, x[pick], y[pick], epochs=4, batch=512, lr=3e-3, seed=2)
        s.graph = _abi.Graph(s.ctx, off, nbr, method=method, dispatch=_abi.DISPATCH_LEARNED)
        s.graph.set_mlp(HIDDEN, params, CAND_THRESH)
    else:
        s.graph = _abi.Graph(s.ctx, off, nbr, method=method)
    return s


def run(s):
    case = s.case
    flow = case["flow"]
    if flow == "train":
        params, loss = _abi.mlp_train(s.ctx, HIDDEN, s.params, s.x, s.y, epochs=case["epochs"], batch=case["batch"],
                                      lr=3e-3, seed=2)
        return {"params": params, "loss": np.float32(loss)}
    if flow == "oneshot":
        with _abi.Graph(s.ctx, s.off, s.nbr, method=METHOD[case["method"]]) as g:
            labels, res = g.run(case["iters"])
        return {"labels": labels, "iterations": res["iterations"]}
    if flow == "steps":
        g, updated = s.graph, []
        g.init()
        for _ in range(case["iters"]):
            st = g.step()
            updated.append(st["updated"])
            if st["stopped"]:
                break
        return {"labels": g.labels(), "updated": updated}
    labels, res = s.graph.run(case["iters"])
    out = {"labels": labels, "iterations": res["iterations"]}
    if flow == "batch":
        out["graph_iterations"] = s.graph.batch_iterations()
    return out


def _sizes(case):
    """Vertices and directed edges, from the generators' parameters."""
    if case["family"] == "pp":
        return case["n"], 2 * case["n"] * (case["intra"] + case["inter"])
    if case["family"] == "rmat":
        return 1 << case["scale"], 2 * case["ef"] << case["scale"]
    if case["family"] == "batch":   # n ~ U[1000, nmax], degree ~ 1.25 U[8, 48]
        n = case["graphs"] * (1000 + case["nmax"]) // 2
        return n, 35 * n
    return case["n"], int(case["avg_deg"] * case["n"])


def work(case):
    if case["flow"] == "train":
        # forward, and backward with respect to activations and weights, of every sample in every epoch; the
        # parameters' Adam state stays on the chip
        params = int(_abi.mlp_num_params(HIDDEN))
        return {"bytes": 20.0 * case["samples"] + 8.0 * params,
                "flops": 6.0 * params * case["samples"] * case["epochs"]}
    n, m = _sizes(case)
    # the graph once (int32 offsets and neighbour ids), the labels out once
    return {"bytes": 4.0 * m + 4.0 * (n + 1) + 4.0 * n, "flops": 0.0}


def exact(case, seed):
    """The training in float64; label propagation's outputs are whole numbers."""
    if case["flow"] != "train":
        return None
    x, y = _samples(case["samples"], seed)
    h, n, b = HIDDEN, case["samples"], min(case["batch"], case["samples"])
    # the seeded shuffle of the samples: Fisher-Yates over a SplitMix64 stream (seed 2)
    mask = (1 << 64) - 1
    step = 0x9E3779B97F4A7C15
    i = np.arange(n - 1, 0, -1, dtype=np.uint64)
    with np.errstate(over="ignore"):
        z = np.uint64((2 ^ 0x5DEECE66D) & mask) + np.uint64(step) * np.arange(1, n, dtype=np.uint64)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    z = (z ^ (z >> np.uint64(31))) % (i + np.uint64(1))
    order = list(range(n))
    for k, j in zip(range(n - 1, 0, -1), z.tolist()):
        order[k], order[j] = order[j], order[k]
    x, y = x[order].astype(np.float64), y[order].astype(np.float64)
    p = _abi.mlp_init(h, seed + 1).astype(np.float64)
    at = np.cumsum([4 * h, h, h * h, h, h, 1])

    def split(q):
        w1, b1, w2, b2, w3, b3 = np.split(q, at[:-1])
        return w1.reshape(h, 4), b1, w2.reshape(h, h), b2, w3, b3

    def forward(xs):
        w1, b1, w2, b2, w3, b3 = split(p)
        h1 = np.maximum(xs @ w1.T + b1, 0.0)
        z2 = h1 @ w2.T + b2
        return h1, z2, np.maximum(z2, 0.0) @ w3 + b3[0]

    mom, var, t = np.zeros_like(p), np.zeros_like(p), 0
    lr, beta1, beta2, eps = (float(np.float32(v)) for v in (3e-3, 0.9, 0.999, 1e-8))
    for _ in range(case["epochs"]):
        for o in range(0, n - b + 1, b):
            xs, ys = x[o:o + b], y[o:o + b]
            h1, z2, out = forward(xs)
            _, _, w2, _, w3, _ = split(p)
            g = (out - ys) / b
            d2 = np.where(z2 > 0, g[:, None] * w3, 0.0)
            d1 = np.where(h1 > 0, d2 @ w2, 0.0)
            grad = np.concatenate([(d1.T @ xs).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0),
                                   np.maximum(z2, 0.0).T @ g, [g.sum()]])
            t += 1
            mom = beta1 * mom + (1 - beta1) * grad
            var = beta2 * var + (1 - beta2) * grad * grad
            p = p - lr * (mom / (1 - beta1 ** t)) / (np.sqrt(var / (1 - beta2 ** t)) + eps)
    loss = float(np.mean(0.5 * (forward(x)[2] - y) ** 2))
    return {"params": p, "loss": np.float64(loss)}
