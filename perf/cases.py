"""The calls that programs built on this package spend their time in, as cases to measure.

A case is one of these calls, at one size:

  linear   one SparseLinear, token-major activations in and out: `train` is forward plus
           backward (input, weight and bias gradients), `infer` forward under no_grad
  mlp      the whole training step of a two-layer MLP classifier (784 -> 512 -> 10 in the
           benchmark): forward, cross-entropy, backward, SGD
  ffn      a transformer block's feed-forward part, SparseLinear -> GELU -> SparseLinear,
           forward plus backward
  matrix   spmm(W, X) on a large PaddedCSR with its backward: long-tailed (Zipf) row lengths,
           as a matrix has after dynamic sparse training, or uniform ones
  set      one SET update of several layers whose transposes are cached: drop, regrow,
           transposes rebuilt
  rigl     one training step of a layer under RigL: forward, backward, SGD, drop, regrow by
           the dense gradient, transposes rebuilt

Activations are N(0, 1), weights have the layer's own initial range. `exact` states the same
calls in 64 bits on dense matrices with plain torch.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import sparsecore_amd as slk
from sparsecore_amd.layout import from_coo, from_dense

DEV = "cuda"
PADDING = 0.2  # the package's default spare capacity per row
LR = 0.01


def listed():
    return [
        # the hidden layer of the MNIST-sized MLP at its training batch: the smallest
        # training call, where launches and host work count
        {"name": "mlp_hidden_train", "kind": "linear", "mode": "train", "k": 784, "m": 512,
         "sparsity": 0.9, "n": 256, "bias": True},
        # that MLP's whole training step, classifier head and optimizer included
        {"name": "mlp_step", "kind": "mlp", "k": 784, "h": 512, "m": 10, "sparsity": 0.9,
         "n": 256},
        # token-by-token generation for eight sequences through the 60M mini-GPT's FFN-up
        {"name": "ffn_up_decode_8", "kind": "linear", "mode": "infer", "k": 768, "m": 3072,
         "sparsity": 0.9, "n": 8, "bias": False},
        # a prompt of arbitrary (odd) length through the same model's fused QKV projection
        {"name": "qkv_prefill_1001", "kind": "linear", "mode": "infer", "k": 768, "m": 2304,
         "sparsity": 0.7, "n": 1001, "bias": False},
        # the 10M char-GPT's QKV projection over its training batch of 8192 tokens
        {"name": "qkv_10m_train", "kind": "linear", "mode": "train", "k": 384, "m": 1152,
         "sparsity": 0.7, "n": 8192, "bias": False},
        # the 60M mini-GPT's QKV projection over its training batch of 8192 tokens
        {"name": "qkv_60m_train", "kind": "linear", "mode": "train", "k": 768, "m": 2304,
         "sparsity": 0.7, "n": 8192, "bias": False},
        # the 60M mini-GPT's feed-forward block over the same batch
        {"name": "ffn_60m_train", "kind": "ffn", "k": 768, "h": 3072, "sparsity": 0.9, "n": 8192},
        # a layer and a batch of packed sequences that fit no tile: ragged in every dimension
        {"name": "ragged_train", "kind": "linear", "mode": "train", "k": 1000, "m": 1537,
         "sparsity": 0.8, "n": 1777, "bias": True},
        # the largest single-GPU layer of the benchmark, at its two sparsities
        {"name": "matrix_16k_95", "kind": "matrix", "m": 16384, "k": 16384, "sparsity": 0.95,
         "n": 4096, "rows": "zipf"},
        {"name": "matrix_16k_99", "kind": "matrix", "m": 16384, "k": 16384, "sparsity": 0.99,
         "n": 4096, "rows": "zipf"},
        # SET's rewrite of one 60M mini-GPT block: QKV, output projection, FFN-up, FFN-down
        {"name": "set_60m_block", "kind": "set", "d": 768, "f": 3072, "blocks": 1},
        # a wide layer's step under RigL with an update in it
        {"name": "rigl_4096", "kind": "rigl", "k": 4096, "m": 4096, "sparsity": 0.95, "n": 4096},
    ]


# ───────────────────────────── drawn cases ─────────────────────────────

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size of [lo, hi]: half the time a multiple of 64 where one fits, else any."""
    v = _log_int(rng, lo, hi)
    if rng.random() < 0.5 and v >= 64:
        v = min(hi, 64 * max(1, round(v / 64)))
    return v


_MOST = 16384 * 16384 * 0.05 * 4096  # slots x columns of the largest listed case


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["matrix"] * 3 + ["mlp", "ffn", "set", "rigl"])
    while True:
        if kind == "linear":
            mode = rng.choice(["train", "train", "infer"])
            c = {"kind": kind, "mode": mode, "k": _size(rng, 64, 4096), "m": _size(rng, 10, 4096),
                 "sparsity": rng.choice([0.7, 0.8, 0.9, 0.95]),
                 "n": _size(rng, 1 if mode == "infer" else 32, 8192),
                 "bias": rng.random() < 0.5}
        elif kind == "matrix":
            c = {"kind": kind, "m": _size(rng, 2048, 16384), "k": _size(rng, 2048, 16384),
                 "sparsity": rng.choice([0.9, 0.95, 0.98, 0.99]), "n": _size(rng, 256, 4096),
                 "rows": rng.choice(["zipf", "uniform"])}
        elif kind == "mlp":
            c = {"kind": kind, "k": _size(rng, 64, 1024), "h": _size(rng, 128, 1024),
                 "m": _size(rng, 10, 100), "sparsity": rng.choice([0.8, 0.9, 0.95]),
                 "n": _size(rng, 32, 1024)}
        elif kind == "ffn":
            d = _size(rng, 256, 1024)
            c = {"kind": kind, "k": d, "h": 4 * d, "sparsity": rng.choice([0.8, 0.9, 0.95]),
                 "n": _size(rng, 256, 8192)}
        elif kind == "set":
            d = _size(rng, 256, 1024)
            c = {"kind": kind, "d": d, "f": 4 * d, "blocks": rng.choice([1, 2])}
        else:
            c = {"kind": kind, "k": _size(rng, 512, 4096), "m": _size(rng, 512, 4096),
                 "sparsity": rng.choice([0.9, 0.95, 0.98]), "n": _size(rng, 256, 8192)}
        if kind != "matrix" or (1 - c["sparsity"]) * c["m"] * c["k"] * c["n"] <= _MOST:
            return c


# ───────────────────────────── inputs ─────────────────────────────

def _gen(seed, part):
    return torch.Generator(device=DEV).manual_seed(seed * 64 + part)


def _normal(shape, seed, part, scale=1.0):
    return torch.randn(shape, generator=_gen(seed, part), device=DEV) * scale


def _fan_in_bound(k, sparsity):
    return 1.0 / math.sqrt(max(1.0, k * (1.0 - sparsity)))


def _keep(counts, k, g):
    """A mask with counts[i] of row i's k columns, each row's a uniform choice. Every seed of a
    case has the same row lengths, so that its arrays have the same sizes."""
    order = torch.rand(counts.numel(), k, generator=g, device=DEV).argsort(dim=1)
    first = torch.arange(k, device=DEV) < counts[:, None]
    return torch.zeros_like(first).scatter_(1, order, first)


def _weights(m, k, sparsity, seed, part):
    """A dense m x k matrix with (1 - sparsity) of its entries kept (binomial row lengths, as a
    random mask gives), uniform in the layer's initial range, and a bias of the same range."""
    g = _gen(seed, part)
    b = _fan_in_bound(k, sparsity)
    draws = torch.randn(m, generator=torch.Generator().manual_seed(m))
    counts = (1.0 - sparsity) * k + math.sqrt(sparsity * (1.0 - sparsity) * k) * draws
    w = torch.empty(m, k, device=DEV).uniform_(-b, b, generator=g)
    w *= _keep(counts.round().clamp(0, k).to(DEV), k, g)
    return w, torch.empty(m, device=DEV).uniform_(-b, b, generator=g)


def _layer(m, k, sparsity, bias, seed, part):
    """A SparseLinear holding _weights, as one loaded from a checkpoint."""
    w, b = _weights(m, k, sparsity, seed, part)
    layer = slk.SparseLinear(k, m, bias=bias, sparsity=sparsity, padding_ratio=PADDING).to(DEV)
    p = from_dense(w, padding_ratio=PADDING)
    sd = {"_values": p.values, "csr_col_indices": p.col_indices, "csr_row_start": p.row_start,
          "csr_row_nnz": p.row_nnz, "csr_row_capacity": p.row_capacity,
          "csr_topology_version": torch.tensor(0)}
    if bias:
        sd["bias"] = b
    layer.load_state_dict(sd)
    return layer


def _row_counts(case):
    """Live slots per row, longest first: Zipf(1.1) row lengths water-filled to the density
    with full rows at the top, or all alike."""
    m, k = case["m"], case["k"]
    total = round((1.0 - case["sparsity"]) * m * k)
    if case["rows"] == "uniform":
        return torch.full((m,), max(1, total // m))
    rank = torch.arange(1, m + 1, dtype=torch.float64) ** -1.1
    lo, hi = 0.0, float(k) * m
    for _ in range(100):
        mid = 0.5 * (lo + hi)
        if (mid * rank).floor().clamp(1, k).sum() < total:
            lo = mid
        else:
            hi = mid
    return (hi * rank).floor().clamp(1, k).long()


def _coordinates(case, seed):
    """(rows, cols, values) of a matrix case: each row's columns a uniform choice."""
    m, k = case["m"], case["k"]
    shuffle = torch.randperm(m, generator=torch.Generator().manual_seed(seed))
    cnt = _row_counts(case)[shuffle].to(DEV)
    g = _gen(seed, 1)
    rows, cols, step = [], [], max(1, (1 << 26) // k)
    for r0 in range(0, m, step):
        r, c = _keep(cnt[r0:r0 + step], k, g).nonzero(as_tuple=True)
        rows.append(r + r0)
        cols.append(c)
    rows, cols = torch.cat(rows), torch.cat(cols)
    return rows, cols, torch.randn(rows.numel(), generator=g, device=DEV) * 0.01


def _set_shapes(case):
    d, f = case["d"], case["f"]
    return [(3 * d, d, 0.7), (d, d, 0.7), (f, d, 0.9), (d, f, 0.9)] * case["blocks"]


def prepare(case, seed):
    kind, n = case["kind"], case.get("n")
    if kind == "linear":
        m, k = case["m"], case["k"]
        train = case["mode"] == "train"
        return {"kind": kind, "train": train,
                "layer": _layer(m, k, case["sparsity"], case["bias"], seed, 1),
                "x": _normal((n, k), seed, 2).requires_grad_(train),
                "dy": _normal((n, m), seed, 3) if train else None}
    if kind == "mlp":
        model = torch.nn.Sequential(
            _layer(case["h"], case["k"], case["sparsity"], True, seed, 1), torch.nn.ReLU(),
            _layer(case["m"], case["h"], case["sparsity"], True, seed, 2))
        return {"kind": kind, "model": model,
                "opt": torch.optim.SGD(model.parameters(), lr=LR),
                "x": torch.rand((n, case["k"]), generator=_gen(seed, 3), device=DEV),
                "labels": torch.randint(0, case["m"], (n,), generator=_gen(seed, 4), device=DEV)}
    if kind == "ffn":
        return {"kind": kind,
                "up": _layer(case["h"], case["k"], case["sparsity"], False, seed, 1),
                "down": _layer(case["k"], case["h"], case["sparsity"], False, seed, 2),
                "x": _normal((n, case["k"]), seed, 3).requires_grad_(),
                "dy": _normal((n, case["k"]), seed, 4)}
    if kind == "matrix":
        rows, cols, vals = _coordinates(case, seed)
        W = from_coo(rows, cols, vals, (case["m"], case["k"]), padding_ratio=PADDING)
        W.values.requires_grad_()
        return {"kind": kind, "W": W, "x": _normal((case["k"], n), seed, 2).requires_grad_(),
                "dy": _normal((case["m"], n), seed, 3)}
    if kind == "set":
        layers = torch.nn.ModuleList(_layer(m, k, s, False, seed, i + 1)
                                     for i, (m, k, s) in enumerate(_set_shapes(case)))
        algo = slk.SET(sparsity=0.9, drop_fraction=0.3, update_freq=1, seed=seed)
        layers.apply(algo)
        for layer in layers:  # training steps before the update have cached every transpose
            x = torch.ones(1024, layer.in_features, device=DEV, requires_grad=True)
            layer(x).sum().backward()
            layer._values.grad = None
        return {"kind": kind, "layers": layers, "algo": algo}
    layer = _layer(case["m"], case["k"], case["sparsity"], False, seed, 1)
    algo = slk.RigL(sparsity=case["sparsity"], drop_fraction=0.3, update_freq=1, seed=seed)
    layer.apply(algo)
    return {"kind": kind, "layer": layer, "algo": algo,
            "opt": torch.optim.SGD(layer.parameters(), lr=LR),
            "x": _normal((n, case["k"]), seed, 2).requires_grad_(),
            "dy": _normal((n, case["m"]), seed, 3, 1.0 / n)}


# ───────────────────────────── one pass ─────────────────────────────

def run(state):
    kind = state["kind"]
    if kind == "linear":
        layer, x = state["layer"], state["x"]
        if not state["train"]:
            with torch.no_grad():
                return layer(x)
        y = layer(x)
        return (y, *torch.autograd.grad(y, [x, *layer.parameters()], state["dy"]))
    if kind == "mlp":
        state["opt"].zero_grad()
        logits = state["model"](state["x"])
        F.cross_entropy(logits, state["labels"]).backward()
        state["opt"].step()
        return (logits.detach(), *(p.detach() for p in state["model"].parameters()))
    if kind == "ffn":
        up, down, x = state["up"], state["down"], state["x"]
        y = down(F.gelu(up(x)))
        return (y, *torch.autograd.grad(y, [x, *up.parameters(), *down.parameters()],
                                        state["dy"]))
    if kind == "matrix":
        W, x = state["W"], state["x"]
        y = slk.spmm(W, x)
        return (y, *torch.autograd.grad(y, [x, W.values], state["dy"]))
    if kind == "set":
        state["algo"].step()
        out = []
        for layer in state["layers"]:
            csr = layer._csr
            out += [csr.values.detach(), csr.col_indices, csr.row_nnz]
        return out
    layer, x = state["layer"], state["x"]
    state["opt"].zero_grad()
    x.grad = None
    y = layer(x)
    y.backward(state["dy"])
    state["opt"].step()
    state["algo"].step()
    csr = layer._csr
    return (y.detach(), x.grad, layer._values.grad, layer._values.detach(), csr.col_indices,
            csr.row_nnz)


# ───────────────────────────── its work, its tolerance ─────────────────────────────

def _capacity(nnz, m):
    return nnz * (1 + PADDING) + 0.5 * m


def _fwd_bytes(nnz, m, k, n):
    return 8 * nnz + 8 * m + 4 * k * n + 4 * m * n


def _train_bytes(nnz, m, k, n):
    """W's slots, X, dY read once; Y, dX and dW (every slot) written once."""
    return 8 * nnz + 8 * m + 4 * (2 * k * n + 2 * m * n) + 4 * _capacity(nnz, m)


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "set":
        b = 0
        for m, k, s in _set_shapes(case):
            cap = _capacity((1 - s) * m * k, m)
            # values and columns read and rewritten, the transpose's values, columns and map
            b += 16 * cap + 16 * _capacity((1 - s) * m * k, k)
        return {"bytes": b, "flops": 0}
    if kind == "mlp":
        d = 1 - case["sparsity"]
        a, b = d * case["h"] * case["k"], d * case["m"] * case["h"]
        return {"bytes": _train_bytes(a, case["h"], case["k"], n) - 4 * case["k"] * n
                + _train_bytes(b, case["m"], case["h"], n) + 4 * (a + b),
                "flops": 4 * a * n + 6 * b * n}
    if kind == "ffn":
        nnz = (1 - case["sparsity"]) * case["k"] * case["h"]
        # the hidden activations and their gradient stay between the two products
        return {"bytes": 2 * _train_bytes(nnz, case["h"], case["k"], n), "flops": 12 * nnz * n}
    m, k = case["m"], case["k"]
    nnz = (1 - case["sparsity"]) * m * k
    if kind == "linear" and case["mode"] == "infer":
        return {"bytes": _fwd_bytes(nnz, m, k, n), "flops": 2 * nnz * n}
    b = _train_bytes(nnz, m, k, n)
    if kind == "rigl":
        # the dense gradient decides the regrowth; the rewrite and the new transpose follow
        return {"bytes": b + 16 * _capacity(nnz, m) + 16 * _capacity(nnz, k),
                "flops": 6 * nnz * n + 2 * m * k * n}
    return {"bytes": b, "flops": 6 * nnz * n}


def tolerance(case):
    """Sums in 32 bits throughout: a few 1e-7 against 64 bits, about 1e-6 with the sums in
    another order. SET moves values and columns and computes none. RigL's regrowth ranks
    rounded sums, so that near ties may fall the other way."""
    if case["kind"] == "set":
        return "exact"
    if case["kind"] == "rigl":
        return {"rel": 1e-5, "differ": 2e-3}
    return {"rel": 1e-5}


# ───────────────────────────── the same in 64 bits ─────────────────────────────

def _slots(w):
    """(rows, cols, slots, total): where each live entry of w is kept in the padded layout."""
    rows, cols = w.nonzero(as_tuple=True)
    nnz = torch.bincount(rows, minlength=w.shape[0])
    cap = (nnz.double() * (1.0 + PADDING)).ceil().clamp(min=1).long()
    start = cap.cumsum(0) - cap
    first = nnz.cumsum(0) - nnz
    slots = start[rows] + torch.arange(rows.numel(), device=w.device) - first[rows]
    return rows, cols, slots, int(cap.sum())


def _padded(dense, where):
    rows, cols, slots, total = where
    out = torch.zeros(total, dtype=torch.float64, device=dense.device)
    out[slots] = dense[rows, cols]
    return out


def exact(case, seed):
    kind, n = case["kind"], case.get("n")
    if kind == "set":
        return None
    if kind == "matrix":
        rows, cols, vals = _coordinates(case, seed)
        w = torch.zeros(case["m"], case["k"], dtype=torch.float64, device=DEV)
        w[rows, cols] = vals.double()
        x = _normal((case["k"], n), seed, 2).double()
        dy = _normal((case["m"], n), seed, 3).double()
        y, dx, where = w @ x, w.t() @ dy, _slots(w)
        del w
        return y, dx, _padded(dy @ x.t(), where)
    if kind == "mlp":
        (w1, b1), (w2, b2) = (_weights(case["h"], case["k"], case["sparsity"], seed, 1),
                              _weights(case["m"], case["h"], case["sparsity"], seed, 2))
        at = _slots(w1), _slots(w2)
        p = [t.double().requires_grad_() for t in (b1, w1, b2, w2)]
        x = torch.rand((n, case["k"]), generator=_gen(seed, 3), device=DEV).double()
        labels = torch.randint(0, case["m"], (n,), generator=_gen(seed, 4), device=DEV)
        logits = F.linear(torch.relu(F.linear(x, p[1], p[0])), p[3], p[2])
        g = torch.autograd.grad(F.cross_entropy(logits, labels), p)
        b1, w1, b2, w2 = [t.detach() - LR * d for t, d in zip(p, g)]
        got = {"_values": (_padded(w1, at[0]), _padded(w2, at[1])), "bias": (b1, b2)}
        names = [name for name, _ in slk.SparseLinear(2, 2).named_parameters()]
        return (logits.detach(), *(got[name][i] for i in (0, 1) for name in names))
    if kind == "ffn":
        w1, _ = _weights(case["h"], case["k"], case["sparsity"], seed, 1)
        w2, _ = _weights(case["k"], case["h"], case["sparsity"], seed, 2)
        at = _slots(w1), _slots(w2)
        x, w1, w2 = (t.double().requires_grad_()
                     for t in (_normal((n, case["k"]), seed, 3), w1, w2))
        y = F.linear(F.gelu(F.linear(x, w1)), w2)
        dx, d1, d2 = torch.autograd.grad(y, [x, w1, w2],
                                         _normal((n, case["k"]), seed, 4).double())
        return y.detach(), dx, _padded(d1, at[0]), _padded(d2, at[1])
    w, b = _weights(case["m"], case["k"], case["sparsity"], seed, 1)
    where = _slots(w)
    w, b = w.double(), b.double()
    x = _normal((n, case["k"]), seed, 2).double()
    if kind == "rigl":
        dy = _normal((n, case["m"]), seed, 3, 1.0 / n).double()
        return x @ w.t(), dy @ w, _padded(dy.t() @ x, where), None, None, None
    y = x @ w.t()
    if case["bias"]:
        y += b
    if case["mode"] == "infer":
        return y
    dy = _normal((n, case["m"]), seed, 3).double()
    got = {"_values": _padded(dy.t() @ x, where), "bias": dy.sum(0)}
    names = [name for name, _ in slk.SparseLinear(2, 2, bias=case["bias"]).named_parameters()]
    return (y, dy @ w, *(got[name] for name in names))
