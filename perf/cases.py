"""The work that a user has the framework do, as measurable cases.

listed() and draw(rng) give cases, prepare(case, seed) what a program holds
before the call (the case's points in the seed's row order), run(state) one pass through the public entry points, work(case)
the bytes and operations the pass cannot do without, exact(case, seed) the
64-bit values of the computed (not counted) outputs.

Kinds:
  run    one clustering call: X on the device (or in host memory, as the
         reference's callers hold it) to labels and subspaces in host memory
  many   many independent data sets in one call (inscy.run_many)
  train  one minibatch step of the learned pruner's network: gradient and Adam
  score  the network's scores of a set of (tree, dimension) pairs
"""

from __future__ import annotations

import itertools
import math
import zlib

import numpy as np
import torch

from gpu_inscy_amd import _lib, datagen, pruner
from gpu_inscy_amd import inscy as INSCY

MODES = {"exact": _lib.MODE_EXACT, "batched": _lib.MODE_BATCHED, "learned": _lib.MODE_LEARNED}


def _run(name, n, d, clusters, lo, hi, sigma, noise, eps, cells, mu, minfrac, **over):
    c = dict(kind="run", n=n, d=d, clusters=clusters, lo=lo, hi=hi, sigma=sigma, noise=noise, zipf=False, eps=eps,
             cells=cells, mu=mu, minfrac=minfrac, rect=True, order=0, mode="batched", host=False)
    c.update(over)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest table a user clusters, of the glass data's shape: launches and read-backs count
        _run("small_table", 214, 9, 4, 3, 6, 0.05, 0.05, 0.01, 4, 8, 0.05, host=True),
        # the base point of the parameter sweeps (experiments.py), a CPU tensor as its harness passes it
        _run("sweep_point", 1500, 15, 4, 12, 12, 0.05, 0.01, 0.01, 4, 8, 0.05, host=True),
        # the reference's CPU/GPU names: the depth-first driver, an odd size
        _run("depth_first", 4999, 11, 6, 3, 7, 0.03, 0.10, 0.015, 6, 4, 0.02, mode="exact"),
        # levels in entropy order (entropy_order = -1, swept by experiments.py as "order")
        _run("entropy_order", 3001, 9, 5, 3, 6, 0.03, 0.10, 0.015, 6, 4, 0.02, order=-1),
        # an ordinary call: n = 25,000, d = 15, 10 clusters
        _run("ordinary", 25000, 15, 10, 4, 8, 0.03, 0.10, 0.015, 6, 4, 0.02),
        # the same size with rectangular=False, the default of every wrapper: the phi density
        _run("ordinary_phi", 24001, 15, 10, 4, 8, 0.03, 0.10, 0.015, 6, 4, 0.02, rect=False),
        # many dimensions (the large-d sweep's parameters, beyond one 64-bit mask word)
        _run("many_dims", 20011, 70, 12, 4, 8, 0.02, 0.05, 0.01, 4, 8, 0.05),
        # many independent data sets in one call
        dict(name="many_sets", kind="many", count=24, n_lo=2000, n_hi=40000, d_lo=8, d_hi=20),
        # the learned pruner's mode on a middle-sized set
        _run("learned", 60000, 20, 14, 4, 9, 0.03, 0.15, 0.02, 8, 4, 0.01, mode="learned"),
        # the benchmark's size: n = 100,000, d = 20, 20 clusters of Zipf sizes
        _run("large", 100000, 20, 20, 4, 10, 0.035, 0.15, 0.02, 8, 4, 0.01, zipf=True),
        # a training step of the pruner's network, the trainer's default minibatch
        dict(name="train_step", kind="train", rows=4096),
        # the scores of a level's pairs
        dict(name="score_pairs", kind="score", rows=200003),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sweep", "ordinary", "ordinary", "phi", "depth", "order", "dims", "many", "learned", "large",
                       "train", "score"])
    if kind == "train":
        return dict(kind="train", rows=_log(rng, 33, 16384))
    if kind == "score":
        return dict(kind="score", rows=_log(rng, 1, 200003))
    if kind == "many":
        lo = _log(rng, 1000, 4000)
        return dict(kind="many", count=rng.randint(3, 24), n_lo=lo, n_hi=_log(rng, lo, 30000), d_lo=rng.randint(5, 8),
                    d_hi=rng.randint(9, 20))
    cells, mu = rng.randint(3, 10), rng.choice([2, 4, 8, 16])
    eps = rng.choice([0.005, 0.01, 0.015, 0.02])
    if kind == "sweep":
        d = rng.randint(5, 20)
        k = max(2, int(0.8 * d))
        return _run(None, _log(rng, 200, 10000), d, rng.randint(2, 8), min(k, 8), min(k, 12), 0.05, 0.01, eps, cells,
                    mu, rng.choice([0.01, 0.05, 0.10]), host=True)
    if kind == "depth":
        return _run(None, _log(rng, 300, 6000), rng.randint(4, 11), rng.randint(2, 6), 3, 6, 0.03, 0.10, eps, cells,
                    mu, 0.02, mode="exact")
    if kind == "order":
        return _run(None, _log(rng, 300, 3500), rng.randint(4, 9), rng.randint(2, 5), 3, 6, 0.03, 0.10, eps, cells,
                    mu, 0.02, order=rng.choice([-1, 1]))
    if kind == "dims":
        return _run(None, _log(rng, 2000, 20000), rng.randint(30, 100), rng.randint(4, 12), 4, 7, 0.02, 0.05, 0.01, 4,
                    8, 0.05)
    if kind == "learned":
        return _run(None, _log(rng, 5000, 50000), rng.randint(10, 20), rng.randint(4, 12), 4, 8, 0.03, 0.15, 0.02, 8,
                    4, 0.01, mode="learned")
    if kind == "large":
        return _run(None, _log(rng, 40000, 90000), rng.randint(14, 20), rng.randint(8, 16), 4, 8, 0.03, 0.15, 0.02, 8,
                    4, 0.01, zipf=rng.random() < 0.5)
    return _run(None, _log(rng, 1000, 40000), rng.randint(6, 18), rng.randint(3, 12), 3, 7,
                round(rng.uniform(0.02, 0.05), 3), 0.10, rng.choice([0.01, 0.015, 0.02]), cells, mu, 0.02,
                rect=kind != "phi")


def _geometry(case):
    """The generator of a case's points: the sizes of a result depend on its data, so a case is one
    set of points, which every seed gives in another row order."""
    return np.random.default_rng(zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode()))


def _clusters(rng, order, n, d, clusters, lo, hi, sigma, noise, zipf):
    X, _, _ = datagen.make_clusters(rng, n, d, clusters, (min(lo, d), min(hi, d)), sigma, noise,
                                    sizes="zipf" if zipf else "equal")
    return torch.from_numpy(X[order.permutation(n)])


def _network_rows(rows, seed):
    """Feature rows of the ranges that the engine's pair features take: fractions and small logarithms."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    X = torch.rand((rows, _lib.MLP_INPUTS), generator=g, device="cuda")
    X[:, 32:] = (X[:, 32:] < 0.15).float()
    y = (torch.rand(rows, generator=g, device="cuda") < 0.25).float()
    w = torch.rand(rows, generator=g, device="cuda") * 1.5 + 0.25
    return X, y, w


def _trainer(seed):
    """The network in the middle of its training: weights, moments, a step number."""
    t = pruner.Trainer(pruner.init_params(seed % 1000))
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    t.m += 1e-3 * torch.randn(t.m.shape, generator=g, device="cuda")
    t.v += 1e-6 * (0.5 + torch.rand(t.v.shape, generator=g, device="cuda"))
    t.step_no = 200
    return t


LR = 1e-3


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        return dict(kind=kind, trainer=_trainer(seed), rows=_network_rows(case["rows"], seed),
                    inv=1.0 / case["rows"])
    if kind == "score":
        w, _, _, _ = pruner.load()
        return dict(kind=kind, trainer=pruner.Trainer(w), rows=_network_rows(case["rows"], seed))
    rng, order = _geometry(case), np.random.default_rng(seed)
    if kind == "many":
        sets = []
        for _ in range(case["count"]):
            n = int(np.exp(rng.uniform(np.log(case["n_lo"]), np.log(case["n_hi"]))))
            d = int(rng.integers(case["d_lo"], case["d_hi"] + 1))
            X = _clusters(rng, order, n, d, int(rng.integers(3, 13)), 3, 8, 0.03, 0.10, False).cuda()
            sets.append((X, 0.015, 1.0, 4, int(0.02 * n), 1.0, 6, True, 0))
        return dict(kind=kind, sets=sets)
    X = _clusters(rng, order, *(case[k] for k in ("n", "d", "clusters", "lo", "hi", "sigma", "noise", "zipf")))
    if not case["host"]:
        X = X.cuda()
    if case["mode"] == "learned":
        pruner.use()
    args = (case["eps"], 1.0, case["mu"], max(1, int(case["n"] * case["minfrac"])), 1.0, case["cells"], case["rect"],
            case["order"])
    return dict(kind=kind, X=X, args=args, mode=MODES[case["mode"]])


def _result(res):
    """The clustering as a program reads it: every subspace's dimensions and every label."""
    subs = res.subspaces
    return {"sizes": np.fromiter((len(s) for s in subs), np.int32, len(subs)),
            "dims": np.fromiter(itertools.chain.from_iterable(subs), np.int32), "labels": res.labels}


def run(state):
    kind = state["kind"]
    if kind == "run":
        return _result(INSCY.run(state["X"], *state["args"], mode=state["mode"]))
    if kind == "many":
        return [_result(r)["labels"] for r in INSCY.run_many(state["sets"])]
    t = state["trainer"]
    X, y, w = state["rows"]
    if kind == "score":
        return t.forward(X)
    g = t.gradient(X, y, w, state["inv"])
    t.adam(LR)
    return {"grad": g, "master": t.master, "m": t.m, "v": t.v}


def work(case):
    kind = case["kind"]
    if kind in ("train", "score"):
        rows, p = case["rows"], _lib.MLP_PARAMS
        macs = _lib.MLP_HIDDEN * (_lib.MLP_INPUTS + _lib.MLP_HIDDEN + 1)
        if kind == "score":
            return {"bytes": rows * (4 * _lib.MLP_INPUTS + 4) + 2 * p, "flops": 2 * macs * rows}
        # weights, moments and gradient once each way; forward, error and weight gradient
        return {"bytes": rows * (4 * _lib.MLP_INPUTS + 8) + 30 * p,
                "flops": 2 * rows * (2 * macs + _lib.MLP_HIDDEN * (_lib.MLP_HIDDEN + 1))}

    def one(n, d, clusters, k, sigma, noise, eps, mu):
        # The input once, a label row per subspace of the result, and per point of each row the
        # distances to its mu core neighbours.  Subspaces: every dimension, and each subset of a
        # cluster's k dimensions in which its points still have mu neighbours (a Gaussian cluster of
        # m points holds about m * ball(L) * (eps / (2 sqrt(pi) sigma))^L of them around a member).
        m, rows = n * (1.0 - noise) / clusters, float(d)
        for L in range(2, min(k, d) + 1):
            ball = math.pi ** (L / 2) / math.gamma(L / 2 + 1)
            if m * ball * (eps / (2.0 * math.sqrt(math.pi) * sigma)) ** L < mu:
                break
            rows += clusters * math.comb(min(k, d), L)
        return 4.0 * n * d + 4.0 * n * rows, 3.0 * 2 * mu * n * rows

    if kind == "many":
        n = (case["n_lo"] * case["n_hi"]) ** 0.5
        b, f = one(n, (case["d_lo"] + case["d_hi"]) // 2, 7.5, 6, 0.03, 0.10, 0.015, 4)
        return {"bytes": case["count"] * b, "flops": case["count"] * f}
    b, f = one(case["n"], case["d"], case["clusters"], (case["lo"] + case["hi"]) // 2, case["sigma"], case["noise"],
               case["eps"], case["mu"])
    return {"bytes": b, "flops": f}


def exact(case, seed):
    """The network's outputs in 64 bits; clusterings are whole numbers and have no value here."""
    if case["kind"] not in ("train", "score"):
        return None
    H, n_in = _lib.MLP_HIDDEN, _lib.MLP_INPUTS
    X, y, w = (t.double() for t in _network_rows(case["rows"], seed))
    if case["kind"] == "score":
        params = torch.from_numpy(pruner.load()[0]).cuda()
    else:
        t = _trainer(seed)
        params = t.master
    q = params.to(torch.bfloat16).double().requires_grad_(case["kind"] == "train")
    cut = np.cumsum([0, H * n_in, H, H * H, H, H, 1])
    W1, b1, W2, b2, w3, b3 = (q[a:b] for a, b in zip(cut[:-1], cut[1:]))
    h = torch.relu(X @ W1.view(H, n_in).t() + b1)
    h = torch.relu(h @ W2.view(H, H).t() + b2)
    z = h @ w3 + b3
    if case["kind"] == "score":
        return torch.sigmoid(z)
    loss = (w * (torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs())) - y * z)).sum() / case["rows"]
    (g,) = torch.autograd.grad(loss, q)
    beta1, beta2 = (float(np.float32(b)) for b in (0.9, 0.999))
    m = beta1 * t.m.double() + (1 - beta1) * g
    v = beta2 * t.v.double() + (1 - beta2) * g * g
    step = t.step_no + 1
    new = t.master.double() - LR * (m / (1 - beta1 ** step)) / (torch.sqrt(v / (1 - beta2 ** step)) + 1e-8)
    return {"grad": torch.cat([g, loss.detach().reshape(1)]), "master": new, "m": m, "v": v}
