"""The work that programs built on this backend have it do, as measurable cases.

Each case is one kind of work at one size:

  mlp            an MLP training loop on the device-resident trainer (MLPTrainer), a span of steps
                 between two reads of the parameters
  dropin         one training step through the reference's own frontend and tape (nn.Sequential,
                 CrossEntropyLoss, SGD / AdamW) on the trait ops, composed or with the fused paths
  linear         one Linear + ReLU layer by itself: the forward product with its epilogue, the input
                 gradient through the ReLU mask below, the weight gradient with the bias gradient
  bmm            a batched product and both of its gradients through transposed views
  loss           softmax cross-entropy with gradient and predictions, then a ReLU backward with the
                 bias gradient, on matrices of one shape
  composed_loss  the reference's op-by-op CrossEntropyLoss, forward and tape backward
  optimizer      one AdamW update over flat buffers or over a list of parameters

A program keeps one Context, as the reference keeps one global backend.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from orcaml_amd import _lib
from orcaml_amd import autodiff as A
from orcaml_amd.backend import HipBackend
from orcaml_amd.device import Context
from orcaml_amd.mlp import MLPTrainer

LR, WD, BETAS, EPS, T0 = 1e-5, 0.01, (0.9, 0.999), 1e-8, 1000
SGD_LR = 1e-4


def listed():
    return [
        # the smallest configuration of the repository: a step is a few launches of microseconds
        {"name": "mlp_small_sgd", "kind": "mlp", "dims": "784,128,128,10", "batch": 64, "opt": "sgd", "steps": 64},
        # the middle configuration: products too small to fill the GPU
        {"name": "mlp_medium_adamw", "kind": "mlp", "dims": "784,1024,1024,10", "batch": 256, "opt": "adamw",
         "steps": 32},
        # the benchmark's configuration
        {"name": "mlp_large_adamw", "kind": "mlp", "dims": "784,4096,4096,10", "batch": 1024, "opt": "adamw",
         "steps": 48},
        # a model nobody padded: odd widths, more classes than the classifier head's kernels take
        {"name": "mlp_ragged_adamw", "kind": "mlp", "dims": "500,1001,333,26", "batch": 200, "opt": "adamw",
         "steps": 32},
        # a layer of a small model at a small batch: latency
        {"name": "linear_small", "kind": "linear", "rows": 32, "in": 256, "out": 256},
        # a layer of odd widths at the last, partial batch of an epoch
        {"name": "linear_ragged", "kind": "linear", "rows": 777, "in": 1003, "out": 1501},
        # a layer that fills the GPU many times over
        {"name": "linear_large", "kind": "linear", "rows": 4096, "in": 4096, "out": 4096},
        # per-sample products over a batch (rank-3 matmul of the trait), an odd length
        {"name": "bmm", "kind": "bmm", "batch": 96, "m": 197, "k": 64, "n": 197},
        # the benchmark's loss and backward epilogue
        {"name": "loss_wide", "kind": "loss", "rows": 8192, "classes": 4096, "onehot": False},
        # the reference's unfused loss on a thousand classes
        {"name": "composed_loss", "kind": "composed_loss", "rows": 1024, "classes": 1000},
        # the benchmark's flat optimizer pass
        {"name": "adamw_flat", "kind": "optimizer", "params": 1 << 28, "segments": 1},
        # a step of the unchanged frontend at the middle configuration: launches and host work
        {"name": "dropin_medium", "kind": "dropin", "dims": "784,1024,1024,10", "batch": 256, "opt": "adamw",
         "fused": False},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, spread over the logarithm; about half are multiples of 8."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and n >= 8:
        n = n // 8 * 8
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "linear", "linear", "linear", "bmm", "loss", "composed_loss", "optimizer",
                       "dropin"])
    if kind == "mlp":
        hidden = [_size(rng, 64, 4096) for _ in range(rng.choice([1, 2, 2, 3]))]
        dims = [_size(rng, 64, 1024)] + hidden + [_size(rng, 2, 200)]
        return {"kind": kind, "dims": ",".join(map(str, dims)), "batch": _size(rng, 8, 1024),
                "opt": rng.choice(["sgd", "adamw"]), "steps": 32}
    if kind == "dropin":
        dims = [_size(rng, 64, 1024), _size(rng, 32, 2048), _size(rng, 32, 2048), _size(rng, 2, 200)]
        return {"kind": kind, "dims": ",".join(map(str, dims)), "batch": _size(rng, 8, 512),
                "opt": rng.choice(["sgd", "adamw"]), "fused": rng.random() < 0.5}
    if kind == "linear":
        return {"kind": kind, "rows": _size(rng, 8, 4096), "in": _size(rng, 32, 4096), "out": _size(rng, 32, 4096)}
    if kind == "bmm":
        m, k, n = (_size(rng, 8, 512) for _ in range(3))
        return {"kind": kind, "batch": _size(rng, 2, min(256, max(4, (1 << 25) // max(m * n, m * k, k * n)))), "m": m,
                "k": k, "n": n}
    if kind == "loss":
        return {"kind": kind, "rows": _size(rng, 8, 8192), "classes": _size(rng, 17, 4096),
                "onehot": rng.random() < 0.5}
    if kind == "composed_loss":
        return {"kind": kind, "rows": _size(rng, 8, 4096), "classes": _size(rng, 2, 2048)}
    return {"kind": kind, "params": _size(rng, 1000, 1 << 27), "segments": rng.choice([1, 1, 4, 6, 12])}


# ---------------------------------------------------------------- inputs
_ctx = None


def _context() -> Context:
    global _ctx
    if _ctx is None:
        _ctx = Context(0)
    return _ctx


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def _dims(case):
    return [int(d) for d in case["dims"].split(",")]


def _onehot(labels, classes):
    return torch.nn.functional.one_hot(labels.long(), classes).float()


def _model(dims, batch, seed):
    """Kaiming-uniform weights, small biases, uniform inputs, uniform labels, and AdamW moments of a run
    that has been going for T0 steps (whose learning rate has decayed: a span of steps then carries
    rounding forward without magnifying it)."""
    g = _gen(seed)
    params, m, v = [], [], []
    for i, o in zip(dims[:-1], dims[1:]):
        params.append((torch.rand((i, o), generator=g, device="cuda") * 2 - 1) / math.sqrt(i))
        params.append(_normal(g, (1, o), 0.01))
    for p in params:
        m.append(_normal(g, p.shape, 1e-3))
        v.append((0.5 + torch.rand(p.shape, generator=g, device="cuda")) * 1e-4)
    x = torch.rand((batch, dims[0]), generator=g, device="cuda")
    labels = torch.randint(0, dims[-1], (batch,), generator=g, device="cuda", dtype=torch.int32)
    return params, m, v, x, labels


def _linear(case, seed):
    """A layer inside a network: x is the ReLU output of the layer below, gy the gradient that has come
    back through this layer's own ReLU."""
    g = _gen(seed)
    r, i, o = case["rows"], case["in"], case["out"]
    x = torch.relu(_normal(g, (r, i)))
    w = (torch.rand((i, o), generator=g, device="cuda") * 2 - 1) / math.sqrt(i)
    b = _normal(g, (1, o), 0.1)
    gy = _normal(g, (r, o), 1e-3) * (torch.rand((r, o), generator=g, device="cuda") < 0.5)
    return x, w, b, gy


def _bmm(case, seed):
    g = _gen(seed)
    b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    return _normal(g, (b, m, k)), _normal(g, (b, k, n), 1 / math.sqrt(k)), _normal(g, (b, m, n), 1e-2)


def _loss(case, seed):
    g = _gen(seed)
    shape = (case["rows"], case["classes"])
    logits = _normal(g, shape, 2.0)
    labels = torch.randint(0, shape[1], (shape[0],), generator=g, device="cuda", dtype=torch.int32)
    return logits, labels, _normal(g, shape), _normal(g, shape, 1e-3)


def _flat(case, seed):
    g = _gen(seed)
    n = case["params"]
    p, grad, m = _normal(g, (n,), 0.02), _normal(g, (n,), 1e-3), _normal(g, (n,), 1e-4)
    v = (0.5 + torch.rand((n,), generator=g, device="cuda")) * 1e-6
    return p, grad, m, v


def _segments(case):
    """(offset, length) of each parameter: weights and biases alternate, as a model's list has them."""
    n, s = case["params"], case["segments"]
    if s == 1:
        return [(0, n)]
    big = (n - (s // 2) * max(1, n // (64 * s))) // (s - s // 2)
    lens = [big if i % 2 == 0 else max(1, n // (64 * s)) for i in range(s)]
    lens[-1] += n - sum(lens)
    out, off = [], 0
    for length in lens:
        out.append((off, length))
        off += length
    return out


def _host(t):
    return t.cpu().numpy()


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    if kind == "mlp":
        dims = _dims(case)
        params, m, v, x, labels = _model(dims, case["batch"], seed)
        adamw = case["opt"] == "adamw"
        tr = MLPTrainer(ctx, dims, case["batch"], kind=case["opt"], lr=LR if adamw else SGD_LR,
                        weight_decay=WD if adamw else 0.0, betas=BETAS, eps=EPS)
        tr.set_params([_host(p) for p in params])
        if adamw:
            tr.set_moments(0, [_host(t) for t in m])
            tr.set_moments(1, [_host(t) for t in v])
            tr.set_step_count(T0)
        tr.set_batch(_host(x), labels=_host(labels))
        return {"kind": kind, "trainer": tr, "steps": case["steps"]}
    if kind == "dropin":
        dims = _dims(case)
        params, m, v, x, labels = _model(dims, case["batch"], seed)
        ad = A.Autodiff(HipBackend(ctx))
        model = A.build_mlp(ad, [_host(p) for p in params])
        if case["opt"] == "adamw":
            opt = A.AdamW(model.parameters(), lr=LR, betas=BETAS, eps=EPS, weight_decay=WD, fused=case["fused"])
            state = {"t": T0}
            for i in range(len(params)):
                state[f"m.{i}"] = A.Tensor.from_numpy(ad, _host(m[i]))
                state[f"v.{i}"] = A.Tensor.from_numpy(ad, _host(v[i]))
            opt.load_state_dict(state)
        else:
            opt = A.SGD(model.parameters(), lr=SGD_LR, fused=case["fused"])
        return {"kind": kind, "ad": ad, "model": model, "opt": opt, "loss": A.CrossEntropyLoss(fused=case["fused"]),
                "x": A.Tensor.from_numpy(ad, _host(x)),
                "target": A.Tensor.from_numpy(ad, _host(_onehot(labels, dims[-1])))}
    if kind == "linear":
        x, w, b, gy = _linear(case, seed)
        y, dx, dw, db = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(w), torch.empty_like(b)
        fwd = _lib.Epilogue(kind=_lib.EPI_BIAS_RELU, bias=b.data_ptr())
        bwd_x = _lib.Epilogue(kind=_lib.EPI_RELU_MASK, mask=x.data_ptr(), ldmask=case["in"])
        bwd_w = _lib.Epilogue(kind=_lib.EPI_NONE, colsum=db.data_ptr())
        return {"kind": kind, "ctx": ctx, "n": (case["rows"], case["in"], case["out"]), "x": x, "w": w, "b": b,
                "gy": gy, "y": y, "dx": dx, "dw": dw, "db": db, "epi": (fwd, bwd_x, bwd_w)}
    if kind == "bmm":
        be = HipBackend(ctx)
        a, b, g = _bmm(case, seed)
        s = [be.from_f32_slice(tuple(t.shape), _host(t)) for t in (a, b, g)]
        return {"kind": kind, "be": be, "s": s, "n": (case["batch"], case["m"], case["k"], case["n"])}
    if kind == "loss":
        logits, labels, pre, grad = _loss(case, seed)
        onehot = _onehot(labels, case["classes"]) if case["onehot"] else None
        rows, classes = logits.shape
        return {"kind": kind, "ctx": ctx, "logits": logits, "labels": labels, "onehot": onehot, "pre": pre,
                "grad": grad, "loss": torch.empty(1, device="cuda"), "dlogits": torch.empty_like(logits),
                "preds": torch.empty(rows, device="cuda", dtype=torch.int32),
                "correct": torch.empty(1, device="cuda", dtype=torch.int64), "dpre": torch.empty_like(pre),
                "db": torch.empty(classes, device="cuda")}
    if kind == "composed_loss":
        ad = A.Autodiff(HipBackend(ctx))
        logits, labels, _, _ = _loss(case, seed)
        return {"kind": kind, "ad": ad, "loss": A.CrossEntropyLoss(),
                "pred": A.Tensor.from_numpy(ad, _host(logits)),
                "target": A.Tensor.from_numpy(ad, _host(_onehot(labels, case["classes"])))}
    p, g, m, v = _flat(case, seed)
    return {"kind": kind, "ctx": ctx, "p": p, "g": g, "m": m, "v": v, "segs": _segments(case), "t": T0}


# ---------------------------------------------------------------- one pass
class _View:
    """A device storage of the backend as another library sees it."""

    def __init__(self, storage, shape):
        self.storage = storage
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (storage.ptr, False),
                                         "version": 2}


def _tensor(storage, shape):
    return torch.as_tensor(_View(storage, shape), device="cuda")


def run(state):
    kind = state["kind"]
    if kind == "mlp":
        tr = state["trainer"]
        for _ in range(state["steps"]):
            tr.step()
        loss, _ = tr.metrics()
        return {"loss": loss, "logits": tr.logits(), "params": tr.params()}
    if kind == "dropin":
        model, opt = state["model"], state["opt"]
        opt.zero_grad()
        logits = model(state["x"])
        loss = state["loss"](logits, state["target"])
        loss.backward()
        grads = [p.tensor.grad() for p in model.parameters()]
        opt.step()
        return {"loss": _tensor(loss.storage.primal, loss.shape),
                "logits": _tensor(logits.storage.primal, logits.shape),
                "grads": [_tensor(g.storage.primal, g.shape) for g in grads],
                "params": [_tensor(p.tensor.storage.primal, p.tensor.shape) for p in model.parameters()]}
    if kind == "linear":
        h, (r, i, o) = state["ctx"].handle, state["n"]
        x, w, gy = state["x"].data_ptr(), state["w"].data_ptr(), state["gy"].data_ptr()
        fwd, bwd_x, bwd_w = state["epi"]
        _lib.call("orca_hip_gemm", h, 0, 0, r, o, i, x, i, w, o, state["y"].data_ptr(), o, ctypes.byref(fwd))
        _lib.call("orca_hip_gemm", h, 0, 1, r, i, o, gy, o, w, o, state["dx"].data_ptr(), i, ctypes.byref(bwd_x))
        _lib.call("orca_hip_gemm", h, 1, 0, i, o, r, x, i, gy, o, state["dw"].data_ptr(), o, ctypes.byref(bwd_w))
        return {k: state[k] for k in ("y", "dx", "dw", "db")}
    if kind == "bmm":
        be, (b, m, k, n) = state["be"], state["n"]
        x, y, g = state["s"]
        out = be.matmul(x, y, (b, m, k), (b, k, n))
        dx = be.matmul(g, be.transpose(y, (b, k, n), 1, 2), (b, m, n), (b, n, k))
        dy = be.matmul(be.transpose(x, (b, m, k), 1, 2), g, (b, k, m), (b, m, n))
        return [_tensor(out, (b, m, n)), _tensor(dx, (b, m, k)), _tensor(dy, (b, k, n))]
    if kind == "loss":
        h = state["ctx"].handle
        rows, classes = state["logits"].shape
        p = {k: t.data_ptr() for k, t in state.items() if isinstance(t, torch.Tensor)}
        _lib.call("orca_hip_softmax_ce", h, p["logits"], rows, classes, p.get("onehot"),
                  None if "onehot" in p else p["labels"], p["loss"], p["dlogits"], p["preds"], p["correct"])
        _lib.call("orca_hip_relu_bw_colsum", h, p["grad"], p["pre"], rows, classes, p["dpre"], p["db"])
        return {k: state[k] for k in ("loss", "dlogits", "preds", "correct", "dpre", "db")}
    if kind == "composed_loss":
        ad, pred = state["ad"], state["pred"]
        ad.tape.clear()
        pred.require_grad()
        loss = state["loss"](pred, state["target"])
        loss.backward()
        return {"loss": _tensor(loss.storage.primal, loss.shape),
                "grad": _tensor(pred.grad().storage.primal, pred.shape)}
    h = state["ctx"].handle
    p, g, m, v = (state[k].data_ptr() for k in "pgmv")
    state["t"] += 1
    if len(state["segs"]) == 1:
        _lib.call("orca_hip_adamw_step", h, p, g, m, v, state["segs"][0][1], LR, *BETAS, EPS, WD, state["t"])
    else:
        table = (_lib.OptSegment * len(state["segs"]))()
        for i, (off, n) in enumerate(state["segs"]):
            o = 4 * off
            table[i] = _lib.OptSegment(p + o, p + o, g + o, m + o, v + o, n)
        _lib.call("orca_hip_adamw_multi", h, table, len(state["segs"]), LR, *BETAS, EPS, WD, state["t"])
    return {k: state[k] for k in ("p", "m", "v")}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("mlp", "dropin"):
        dims, b, steps = _dims(case), case["batch"], case.get("steps", 1)
        macs = sum(i * o for i, o in zip(dims[:-1], dims[1:]))
        params = macs + sum(dims[1:])
        flops = 2 * b * (3 * macs - dims[0] * dims[1])
        moved = params * (24 if case["opt"] == "adamw" else 8) + 4 * b * (dims[0] + 2 * dims[-1])
        return {"bytes": steps * moved, "flops": steps * flops}
    if kind == "linear":
        r, i, o = case["rows"], case["in"], case["out"]
        return {"bytes": 4 * (r * i + i * o + o + r * o + r * o + r * i + i * o + o), "flops": 6 * r * i * o}
    if kind == "bmm":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        return {"bytes": 8 * b * (m * k + k * n + m * n), "flops": 6 * b * m * k * n}
    if kind == "loss":
        r, c = case["rows"], case["classes"]
        return {"bytes": 4 * r * c * (6 if case["onehot"] else 5) + 8 * r + 4 * c, "flops": 12 * r * c}
    if kind == "composed_loss":
        r, c = case["rows"], case["classes"]
        return {"bytes": 12 * r * c, "flops": 12 * r * c}
    return {"bytes": 28 * case["params"], "flops": 15 * case["params"]}


def tolerance(case):
    """About four times the error against 64 bits that was measured, where nothing more than rounding is in
    play.  A whole model adds ReLU masks: a pre-activation within rounding of zero may be masked or not, which
    changes one column of a weight gradient by one sample's share (about 2e-3 of its norm at 784-1024-1024-10,
    256 rows) and, diluted by the step size, the parameters after a span of steps."""
    kind = case["kind"]
    if kind == "mlp":  # 4e-6 measured without such a difference
        return {"rel": 2e-4, "max": 5e-2}
    if kind == "dropin":  # gradients of one step; 4e-7 measured without
        return {"rel": 2e-3, "max": 3e-1}
    if kind == "linear":  # 8e-7 at 4096 terms
        return {"rel": 4e-6, "max": 5e-5}
    if kind == "bmm":  # 4e-7 at 512 terms
        return {"rel": 2e-6, "max": 2e-5}
    if kind in ("loss", "composed_loss"):  # 5e-7
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 2e-7, "max": 2e-6}  # element by element: 4e-8


# ---------------------------------------------------------------- the same in 64 bits
def _mlp_step64(dims, params, x, labels):
    """Loss, logits and gradients of one forward and backward pass."""
    hs, h = [x], x
    n = len(dims) - 1
    for l in range(n):
        h = h @ params[2 * l] + params[2 * l + 1]
        if l + 1 < n:
            h = torch.relu(h)
            hs.append(h)
    logits = h
    logp = torch.log_softmax(logits, 1)
    idx = labels.long()[:, None]
    loss = -logp.gather(1, idx).mean()
    d = torch.exp(logp)
    d.scatter_add_(1, idx, torch.full(idx.shape, -1.0, dtype=d.dtype, device=d.device))
    d /= x.shape[0]
    grads = [None] * (2 * n)
    for l in range(n - 1, -1, -1):
        grads[2 * l] = hs[l].t() @ d
        grads[2 * l + 1] = d.sum(0, keepdim=True)
        if l:
            d = (d @ params[2 * l].t()) * (hs[l] > 0)
    return loss, logits, grads


def _adamw64(p, g, m, v, t):
    m = BETAS[0] * m + (1 - BETAS[0]) * g
    v = BETAS[1] * v + (1 - BETAS[1]) * g * g
    mh, vh = m / (1 - BETAS[0] ** t), v / (1 - BETAS[1] ** t)
    return p * (1 - LR * WD) - LR * mh / (vh.sqrt() + EPS), m, v


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mlp", "dropin"):
        dims = _dims(case)
        params, m, v, x, labels = _model(dims, case["batch"], seed)
        params, m, v, x = [p.double() for p in params], [t.double() for t in m], [t.double() for t in v], x.double()
        for s in range(case.get("steps", 1)):
            loss, logits, grads = _mlp_step64(dims, params, x, labels)
            for i, g in enumerate(grads):
                if case["opt"] == "adamw":
                    params[i], m[i], v[i] = _adamw64(params[i], g, m[i], v[i], T0 + 1 + s)
                else:
                    params[i] = params[i] - SGD_LR * g
        if kind == "mlp":
            return {"loss": float(loss), "logits": logits, "params": params}
        return {"loss": loss.reshape(1), "logits": logits, "grads": grads, "params": params}
    if kind == "linear":
        x, w, b, gy = (t.double() for t in _linear(case, seed))
        return {"y": torch.relu(x @ w + b), "dx": (gy @ w.t()) * (x > 0), "dw": x.t() @ gy,
                "db": gy.sum(0, keepdim=True)}
    if kind == "bmm":
        a, b, g = (t.double() for t in _bmm(case, seed))
        return [torch.matmul(a, b), torch.matmul(g, b.transpose(1, 2).contiguous()),
                torch.matmul(a.transpose(1, 2).contiguous(), g)]
    if kind in ("loss", "composed_loss"):
        logits, labels, pre, grad = _loss(case, seed)
        x, idx = logits.double(), labels.long()[:, None]
        logp = torch.log_softmax(x, 1)
        loss = -logp.gather(1, idx).mean().reshape(1)
        d = torch.exp(logp)
        d.scatter_add_(1, idx, torch.full(idx.shape, -1.0, dtype=d.dtype, device=d.device))
        d /= x.shape[0]
        if kind == "composed_loss":
            return {"loss": loss, "grad": d}
        dpre = grad.double() * (pre > 0)
        return {"loss": loss, "dlogits": d, "preds": None, "correct": None, "dpre": dpre, "db": dpre.sum(0)}
    p, g, m, v = (t.double() for t in _flat(case, seed))
    p, m, v = _adamw64(p, g, m, v, T0 + 1)
    return {"p": p, "m": m, "v": v}
