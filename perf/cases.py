"""Performance cases: the work a user has this backend do, through its public entry points.

Kinds of case (the "kind" entry):
  train      one optimizer step of a device-resident training session (HipTrainingSession):
             forward, loss, backward and the transactional update; with "micro" > 1 the step
             accumulates that many micro-batches first (GradientMode.ACCUMULATE / _AND_STEP);
  infer      the forward program of a Linear chain (lower_forward): batch-1 calls and batches;
  layer      one Linear layer forward and backward with an upstream cotangent
             (lower_dense_layer): a block of a larger model;
  softmax    a program of row softmax or log-softmax with log-sum-exp and the mean over the rows,
             and for softmax the backward pass with the log-sum-exp cotangent folded in;
  loss       index cross-entropy over many classes with its gradient;
  partition  a planned partition through the backend SPI (analyze, finalize, bind, execute):
             column statistics, a broadcast elementwise chain and row reductions.

Inputs, weights and outputs are in GPU memory when a pass begins, as a training loop or a server
keeps them; a pass is the synchronous call a program makes.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from synaptik_amd.backend import HipBackendIntegration, Node, Partition, TensorDescriptor
from synaptik_amd.native import HipBuffer, HipProgram
from synaptik_amd.program import ProgramBuilder
from synaptik_amd.training import (Adam, AdamW, GradientMode, HipTrainingSession, MlpSpec, Sgd,
                                   TrainingState, lower_dense_layer, lower_forward)

STEPS_BEFORE = 10  # completed optimizer steps of the training state a pass continues from
MAX_FLOPS = 1.9e12  # of a drawn case
MAX_BYTES = 5.0e9


def listed():
    return [
        # The plumbing MLP of the tests and the benchmark: every launch is tiny, latency is all.
        dict(name="train_tiny", kind="train", widths="16-64-1", act="tanh", loss="mse",
             optimizer="sgd", batch=256, labels="i64", micro=1),
        # The benchmark's digit classifier with Adam: mid-size GEMMs and a ten-class head.
        dict(name="train_classifier", kind="train", widths="784-1024-1024-10", act="relu",
             loss="ce", optimizer="adam", batch=1024, labels="i64", micro=1),
        # A classifier whose widths are what its data gave it: nothing is a multiple of anything.
        dict(name="train_ragged", kind="train", widths="617-1021-509-101", act="tanh", loss="ce",
             optimizer="adamw", batch=500, labels="i32", micro=1),
        # A regressor trained with gradient accumulation over two micro-batches.
        dict(name="train_accumulate", kind="train", widths="512-1024-512-64", act="tanh",
             loss="mse", optimizer="nesterov", batch=128, labels="i64", micro=2),
        # The benchmark's headline network: large square GEMMs.
        dict(name="train_mlp4096", kind="train", widths="4096-4096-4096-4096-4096-4096",
             act="relu", loss="mse", optimizer="momentum", batch=4096, labels="i64", micro=1),
        # One request at a time through the trained digit classifier.
        dict(name="infer_single", kind="infer", widths="784-1024-1024-10", act="relu", batch=1),
        # A server's batch through a wider network: few rows, large weights.
        dict(name="infer_batch", kind="infer", widths="1024-4096-4096-1000", act="relu", batch=64),
        # The benchmark's fused layer, forward and backward.
        dict(name="layer_fused", kind="layer", batch=8192, fan_in=1024, fan_out=1024, act="relu",
             layout="in_out"),
        # A layer of odd extents in Linear's own weight layout.
        dict(name="layer_ragged", kind="layer", batch=3001, fan_in=1531, fan_out=2047, act="tanh",
             layout="out_in"),
        # The benchmark's softmax stress: rows of a power of two, twice the caches' size and more.
        dict(name="softmax_rows", kind="softmax", rows=65536, cols=4096, log=False),
        # A vocabulary's cross-entropy and its gradient; padded positions are ignored.
        dict(name="loss_vocabulary", kind="loss", rows=4096, classes=32003, labels="i64",
             ignore=True),
        # Feature standardisation, scaling, activation and row statistics of a table.
        dict(name="partition_table", kind="partition", rows=20000, cols=1001, act="TANH"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """An extent of the range: as drawn (often odd), or rounded to what a person would type."""
    w = _log_int(rng, lo, hi)
    step = rng.choice([1, 1, 4, 16, 64])
    return max(lo, w // step * step)


def draw(rng):
    kind = rng.choice(["train", "train", "train", "infer", "layer", "layer", "softmax", "loss",
                       "partition"])
    while True:
        if kind == "train":
            loss = rng.choice(["mse", "ce"])
            hidden = [_width(rng, 16, 4096) for _ in range(rng.randint(1, 4))]
            last = _width(rng, 2, 1000) if loss == "ce" else _width(rng, 1, 4096)
            case = dict(kind=kind, widths="-".join(map(str, [_width(rng, 8, 4096)] + hidden + [last])),
                        act=rng.choice(["relu", "tanh", "sigmoid"]), loss=loss,
                        optimizer=rng.choice(["sgd", "momentum", "nesterov", "adam", "adamw"]),
                        batch=_width(rng, 32, 4096), labels=rng.choice(["i32", "i64"]),
                        micro=rng.choice([1, 1, 1, 2]))
        elif kind == "infer":
            hidden = [_width(rng, 64, 4096) for _ in range(rng.randint(1, 4))]
            case = dict(kind=kind, widths="-".join(map(str, [_width(rng, 16, 4096)] + hidden
                                                        + [_width(rng, 1, 1000)])),
                        act=rng.choice(["relu", "tanh", "sigmoid"]), batch=_width(rng, 1, 4096))
        elif kind == "layer":
            case = dict(kind=kind, batch=_width(rng, 64, 8192), fan_in=_width(rng, 64, 4096),
                        fan_out=_width(rng, 64, 4096), act=rng.choice(["relu", "tanh", "sigmoid"]),
                        layout=rng.choice(["in_out", "out_in"]))
        elif kind == "softmax":
            case = dict(kind=kind, rows=_width(rng, 64, 65536), cols=_width(rng, 10, 32768),
                        log=rng.choice([False, False, True]))
        elif kind == "loss":
            case = dict(kind=kind, rows=_width(rng, 64, 16384), classes=_width(rng, 17, 50000),
                        labels=rng.choice(["i32", "i64"]), ignore=rng.choice([False, True]))
        else:
            case = dict(kind=kind, rows=_width(rng, 64, 65536), cols=_width(rng, 8, 4096),
                        act=rng.choice(["RELU", "TANH", "SIGMOID"]))
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


# ---- what a program has in hand: one backend for the process, torch tensors bound to it ----
_backend = None


def _integration():
    global _backend
    if _backend is None:
        _backend = HipBackendIntegration.open(0)
    return _backend


def _bind(t):
    """The tensor's memory as a buffer of the backend's context."""
    return HipBuffer(_integration().context, t.numel() * t.element_size(), t.data_ptr())


class _Memory:
    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, version=2,
                                             data=(buf.device_pointer(), False))


def _tensor(buf, shape):
    """A float32 buffer of the backend as a tensor over the same memory; the tensor keeps the
    buffer alive, as the session that owns it may go first."""
    t = torch.as_tensor(_Memory(buf, shape, "<f4"), device="cuda")
    t.buffer = buf
    return t


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)


def _normal(g, shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(scale)


def _empty(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.float32)


def _chain(case):
    w = [int(x) for x in case["widths"].split("-")]
    return list(zip(w, w[1:]))


def _parameters(case, g):
    """Glorot-scaled weights and small biases, as some way into training."""
    Ws = [_normal(g, (o, i), math.sqrt(2.0 / (i + o))) for i, o in _chain(case)]
    bs = [_normal(g, (o,), 0.05) for _, o in _chain(case)]
    return Ws, bs


LEARNING = dict(lr=1e-3, momentum=0.9, beta1=0.9, beta2=0.999, eps=1e-8, decay=1e-2)


def _optimizer(case):
    k = LEARNING
    return {"sgd": lambda: Sgd(k["lr"]),
            "momentum": lambda: Sgd(k["lr"], momentum=k["momentum"]),
            "nesterov": lambda: Sgd(k["lr"], momentum=k["momentum"], nesterov=True),
            "adam": lambda: Adam(k["lr"]),
            "adamw": lambda: AdamW(k["lr"], weight_decay=k["decay"])}[case["optimizer"]]()


def _training_inputs(case, seed):
    """Weights, biases, optimizer slots and micro-batches of a training case."""
    g = _generator(seed)
    Ws, bs = _parameters(case, g)
    params = Ws + bs
    n = case["batch"]
    fan_in, fan_out = _chain(case)[0][0], _chain(case)[-1][1]
    first, second = [], []
    if case["optimizer"] != "sgd":
        # slots of the size that gradients of such a network leave behind
        first = [_normal(g, p.shape, 1e-3) for p in params]
    if case["optimizer"] in ("adam", "adamw"):
        second = [_normal(g, p.shape, 1e-3).square_().add_(1e-7) for p in params]
    batches = []
    for _ in range(case["micro"]):
        x = _normal(g, (n, fan_in))
        if case["loss"] == "mse":
            y = _normal(g, (n, fan_out))
        else:
            y = torch.randint(0, fan_out, (n,), generator=g, device="cuda",
                              dtype=torch.int32 if case["labels"] == "i32" else torch.int64)
        batches.append((x, y))
    return Ws, bs, first, second, batches


def _prepare_train(case, seed):
    Ws, bs, first, second, batches = _training_inputs(case, seed)
    host = [[t.cpu().numpy() for t in ts] for ts in (Ws, bs, first, second)]
    spec = MlpSpec.chain([int(x) for x in case["widths"].split("-")], hidden=case["act"],
                         loss=case["loss"])
    sess = HipTrainingSession.open(_integration().context, spec, host[0], host[1],
                                   _optimizer(case), case["batch"], label_dtype=case["labels"])
    sess.restore(TrainingState(host[0], host[1], host[2], host[3], STEPS_BEFORE))
    bound = [(_bind(x), _bind(y)) for x, y in batches]
    return dict(kind="train", session=sess, batches=bound, tensors=batches, views={},
                loss=_tensor(sess.loss, (1,)), shapes=[(tuple(t.shape)) for t in Ws + bs])


def _run_train(s):
    sess, batches = s["session"], s["batches"]
    if len(batches) == 1:
        sess.run_resident(*batches[0])
    else:
        for x, y in batches[:-1]:
            sess.run_resident(x, y, GradientMode.ACCUMULATE)
        sess.run_resident(*batches[-1], GradientMode.ACCUMULATE_AND_STEP)
    # the session's current buffers (two sets alternate) as tensors
    current = sess.W[0].handle.value
    views = s["views"].get(current)
    if views is None:
        shapes = s["shapes"]
        views = s["views"][current] = dict(
            loss=s["loss"], parameters=[_tensor(b, q) for b, q in zip(sess.W + sess.b, shapes)],
            first=[_tensor(b, q) for b, q in zip(sess.first, shapes)],
            second=[_tensor(b, q) for b, q in zip(sess.second, shapes)])
    return views


def _activate(act, z):
    return {"relu": torch.relu, "tanh": torch.tanh, "sigmoid": torch.sigmoid}[act](z)


def _forward64(Ws, bs, x, act):
    for i, (W, b) in enumerate(zip(Ws, bs)):
        x = x @ W.t() + b
        if i < len(Ws) - 1:
            x = _activate(act, x)
    return x


def _exact_train(case, seed):
    Ws, bs, first, second, batches = _training_inputs(case, seed)
    params = [p.double().requires_grad_() for p in Ws + bs]
    L = len(Ws)
    total = [torch.zeros_like(p) for p in params]
    for x, y in batches:
        out = _forward64(params[:L], params[L:], x.double(), case["act"])
        if case["loss"] == "mse":
            loss = (out - y.double()).square().mean()
        else:
            loss = torch.nn.functional.cross_entropy(out, y.long())
        for t, d in zip(total, torch.autograd.grad(loss, params)):
            t += d
    f32 = lambda v: float(np.float32(v))  # noqa: E731
    k = {n: f32(v) for n, v in LEARNING.items()}
    new, m1, m2 = [], [], []
    with torch.no_grad():
        for i, (p, g) in enumerate(zip(params, total)):
            if case["optimizer"] in ("adam", "adamw"):
                step = STEPS_BEFORE + 1
                m = k["beta1"] * first[i].double() + (1 - k["beta1"]) * g
                v = k["beta2"] * second[i].double() + (1 - k["beta2"]) * g * g
                base = p * (1 - k["lr"] * k["decay"]) if case["optimizer"] == "adamw" else p
                m1.append(m)
                m2.append(v)
                new.append(base - k["lr"] * (m / (1 - k["beta1"] ** step))
                           / ((v / (1 - k["beta2"] ** step)).sqrt() + k["eps"]))
            elif case["optimizer"] == "sgd":
                new.append(p - k["lr"] * g)
            else:
                m = k["momentum"] * first[i].double() + g
                m1.append(m)
                new.append(p - k["lr"] * (g + k["momentum"] * m if case["optimizer"] == "nesterov"
                                          else m))
    return dict(loss=loss.detach().reshape(1), parameters=[p.detach() for p in new], first=m1,
                second=m2)


# ---- inference ----
def _infer_inputs(case, seed):
    g = _generator(seed)
    Ws, bs = _parameters(case, g)
    return Ws, bs, _normal(g, (case["batch"], _chain(case)[0][0]))


def _prepare_infer(case, seed):
    Ws, bs, x = _infer_inputs(case, seed)
    spec = MlpSpec.chain([int(w) for w in case["widths"].split("-")], hidden=case["act"])
    prog = HipProgram(_integration().context, lower_forward(spec, case["batch"]).image())
    out = _empty(case["batch"], _chain(case)[-1][1])
    ins = Ws + bs + [x]
    return dict(kind="infer", program=prog, keep=ins, out=out,
                bound=prog.bind([_bind(t) for t in ins], [_bind(out)]))


def _exact_infer(case, seed):
    Ws, bs, x = _infer_inputs(case, seed)
    return _forward64([w.double() for w in Ws], [b.double() for b in bs], x.double(), case["act"])


# ---- one layer ----
def _layer_inputs(case, seed):
    g = _generator(seed)
    B, I, O = case["batch"], case["fan_in"], case["fan_out"]
    W = _normal(g, (I, O) if case["layout"] == "in_out" else (O, I), math.sqrt(2.0 / (I + O)))
    return _normal(g, (B, I)), W, _normal(g, (O,), 0.05), _normal(g, (B, O), 1.0 / B)


def _prepare_layer(case, seed):
    ins = _layer_inputs(case, seed)
    B, I, O = case["batch"], case["fan_in"], case["fan_out"]
    pb, _ = lower_dense_layer(B, I, O, case["act"], case["layout"])
    prog = HipProgram(_integration().context, pb.image())
    outs = [_empty(B, O), _empty(B, I), _empty(*ins[1].shape), _empty(O)]
    return dict(kind="layer", program=prog, keep=ins, out=outs,
                bound=prog.bind([_bind(t) for t in ins], [_bind(t) for t in outs]))


def _exact_layer(case, seed):
    x, W, b, dy = (t.double() for t in _layer_inputs(case, seed))
    in_out = case["layout"] == "in_out"
    y = _activate(case["act"], x @ (W if in_out else W.t()) + b)
    slope = {"relu": lambda: (y > 0).double(), "tanh": lambda: 1 - y * y,
             "sigmoid": lambda: y * (1 - y)}[case["act"]]()
    dz = dy * slope
    dx = dz @ (W.t() if in_out else W)
    dW = x.t() @ dz if in_out else dz.t() @ x
    return [y, dx, dW, dz.sum(0)]


# ---- softmax ----
def _softmax_inputs(case, seed):
    g = _generator(seed)
    x = _normal(g, (case["rows"], case["cols"]), 3.0)
    # a few outliers of +-30, as the benchmark's stress has
    at = torch.randint(0, case["cols"], (case["rows"], 2), generator=g, device="cuda")
    x.scatter_(1, at[:, :1], 30.0)
    x.scatter_(1, at[:, 1:], -30.0)
    return x, None if case["log"] else _normal(g, x.shape)


def _prepare_softmax(case, seed):
    x, dp = _softmax_inputs(case, seed)
    R, C = case["rows"], case["cols"]
    pb = ProgramBuilder()
    sx = pb.input(R * C)
    sdp = pb.input(R * C) if dp is not None else None
    sp, sl, sm = pb.output(R * C), pb.output(R), pb.output(1)
    pb.softmax(sx, sp, R, C, lse=sl, log=case["log"])
    pb.reduce_all(sl, sm, R, "mean")
    ins, outs = [x], [_empty(R, C), _empty(R), _empty(1)]
    if dp is not None:
        sdx = pb.output(R * C)
        pb.softmax_bwd(sp, sdp, sdx, R, C, rowscale_const=1.0 / R)
        ins.append(dp)
        outs.append(_empty(R, C))
    prog = HipProgram(_integration().context, pb.image())
    return dict(kind="softmax", program=prog, keep=ins, out=outs,
                bound=prog.bind([_bind(t) for t in ins], [_bind(t) for t in outs]))


def _exact_softmax(case, seed):
    x, dp = _softmax_inputs(case, seed)
    if x.numel() > 1 << 28:
        return None  # six arrays in 64 bits of this size do not fit beside the rest
    x = x.double()
    lse = torch.logsumexp(x, 1)
    if dp is None:
        return [x - lse[:, None], lse, lse.mean().reshape(1)]
    p = torch.softmax(x, 1)
    d = dp.double()
    return [p, lse, lse.mean().reshape(1),
            p * (d - (d * p).sum(1, keepdim=True)) + p * float(np.float32(1.0 / case["rows"]))]


# ---- index cross-entropy ----
IGNORED = -100


def _loss_inputs(case, seed):
    g = _generator(seed)
    R, C = case["rows"], case["classes"]
    z = _normal(g, (R, C), 2.0)
    t = torch.randint(0, C, (R,), generator=g, device="cuda",
                      dtype=torch.int32 if case["labels"] == "i32" else torch.int64)
    if case["ignore"]:
        t[torch.rand((R,), generator=g, device="cuda") < 0.1] = IGNORED
    return z, t


def _prepare_loss(case, seed):
    z, t = _loss_inputs(case, seed)
    R, C = case["rows"], case["classes"]
    pb = ProgramBuilder()
    sz, st = pb.input(R * C), pb.input(R, case["labels"])
    sl, sg = pb.output(1), pb.output(R * C)
    pb.index_ce(sz, st, sl, R, C, grad=sg, ignore_index=IGNORED if case["ignore"] else None)
    prog = HipProgram(_integration().context, pb.image())
    outs = [_empty(1), _empty(R, C)]
    return dict(kind="loss", program=prog, keep=[z, t], out=outs,
                bound=prog.bind([_bind(z), _bind(t)], [_bind(o) for o in outs]))


def _exact_loss(case, seed):
    z, t = _loss_inputs(case, seed)
    z, t = z.double(), t.long()
    kept = t != IGNORED
    n = kept.sum().double()
    safe = t.clamp(min=0)
    lse = torch.logsumexp(z, 1)
    loss = ((lse - z.gather(1, safe[:, None])[:, 0]) * kept).sum() / n
    grad = torch.exp(z - lse[:, None])
    grad.scatter_add_(1, safe[:, None], torch.full_like(grad[:, :1], -1.0))
    return [loss.reshape(1), grad * (kept.double() / n)[:, None]]


# ---- a partition through the SPI ----
EPSILON = 1e-5


def _partition(case):
    R, C = case["rows"], case["cols"]
    f = lambda *s: TensorDescriptor("FLOAT32", tuple(s))  # noqa: E731
    full, row, col = f(R, C), f(C), f(R)
    values = {"x": full, "gamma": row, "beta": row}
    nodes = []

    def node(kind, out, desc, *ins, **attrs):
        values[out] = desc
        nodes.append(Node(kind, list(ins), out, attrs))
        return out

    mean = node("EXPAND", "mean_all", full, node("MEAN", "mean", row, "x", axes=(0,)))
    d = node("SUB", "d", full, "x", mean)
    var = node("MEAN", "var", row, node("MUL", "sq", full, d, d), axes=(0,))
    eps = node("CONSTANT", "eps", row, value=EPSILON)
    sd = node("SQRT", "sd", row, node("ADD", "var_eps", row, var, eps))
    z = node("DIV", "z", full, d, node("EXPAND", "sd_all", full, sd))
    zg = node("MUL", "zg", full, z, node("EXPAND", "gamma_all", full, "gamma"))
    zb = node("ADD", "zb", full, zg, node("EXPAND", "beta_all", full, "beta"))
    a = node(case["act"], "a", full, zb)
    node("MAX", "row_max", col, a, axes=(1,))
    node("MEAN", "row_mean", col, a, axes=(1,))
    node("LOG_SUM_EXP", "row_lse", col, a, axis=1)
    node("SUM", "total", f(), a)
    return Partition(values, nodes, ["x", "gamma", "beta"],
                     ["a", "row_max", "row_mean", "row_lse", "total"])


def _partition_inputs(case, seed):
    g = _generator(seed)
    C = case["cols"]
    x = _normal(g, (case["rows"], C)) * (0.5 + torch.rand((C,), generator=g, device="cuda"))
    x += _normal(g, (C,))
    return x, 1.0 + _normal(g, (C,), 0.1), 0.5 + _normal(g, (C,), 0.1)


def _prepare_partition(case, seed):
    ins = _partition_inputs(case, seed)
    exe = _integration().prepare(_partition(case))
    R, C = case["rows"], case["cols"]
    outs = [_empty(R, C), _empty(R), _empty(R), _empty(R), _empty(1)]
    bound = exe.bind({v: _bind(t) for v, t in zip(("x", "gamma", "beta"), ins)},
                     [_bind(t) for t in outs])
    return dict(kind="partition", executable=exe, bound=bound, keep=ins, out=outs)


def _exact_partition(case, seed):
    x, gamma, beta = (t.double() for t in _partition_inputs(case, seed))
    d = x - x.mean(0)
    sd = (d.square().mean(0) + float(np.float32(EPSILON))).sqrt()
    a = _activate(case["act"].lower(), d / sd * gamma + beta)
    return [a, a.max(1).values, a.mean(1), torch.logsumexp(a, 1), a.sum().reshape(1)]


_PREPARE = dict(train=_prepare_train, infer=_prepare_infer, layer=_prepare_layer,
                softmax=_prepare_softmax, loss=_prepare_loss, partition=_prepare_partition)
_EXACT = dict(train=_exact_train, infer=_exact_infer, layer=_exact_layer, softmax=_exact_softmax,
              loss=_exact_loss, partition=_exact_partition)


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()  # the tensors are written before another stream reads them
    return state


def run(state):
    if state["kind"] == "train":
        return _run_train(state)
    if state["kind"] == "partition":
        state["bound"].execute()
    else:
        state["program"].run_bound(state["bound"])
    return state["out"]


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def work(case):
    """Bytes: inputs read once, outputs and updated state written once. Operations: two for each
    multiply-add of the matrix products (three products for each trained layer, two for the
    first), a few for each element of the rest."""
    kind = case["kind"]
    if kind in ("train", "infer"):
        chain = _chain(case)
        params = sum(i * o + o for i, o in chain)
        products = 2.0 * sum(i * o for i, o in chain)
        n = case["batch"]
        ends = n * (chain[0][0] + chain[-1][1])
        if kind == "infer":
            return {"bytes": 4.0 * (params + ends), "flops": products * n}
        slots = {"sgd": 0, "momentum": 1, "nesterov": 1, "adam": 2, "adamw": 2}[case["optimizer"]]
        samples = n * case["micro"]
        return {"bytes": 4.0 * (2 * (1 + slots) * params + ends * case["micro"]),
                "flops": samples * (3 * products - 2.0 * chain[0][0] * chain[0][1])}
    if kind == "layer":
        B, I, O = case["batch"], case["fan_in"], case["fan_out"]
        return {"bytes": 4.0 * (2 * B * I + 2 * B * O + 2 * I * O + 2 * O), "flops": 6.0 * B * I * O}
    if kind == "softmax":
        n = float(case["rows"]) * case["cols"]
        return {"bytes": 4.0 * n * (2 if case["log"] else 4), "flops": n * (4 if case["log"] else 8)}
    if kind == "loss":
        n = float(case["rows"]) * case["classes"]
        return {"bytes": 8.0 * n, "flops": 6.0 * n}
    n = float(case["rows"]) * case["cols"]
    return {"bytes": 8.0 * n, "flops": 14.0 * n}


def tolerance(case):
    """About four times the largest relative error against 64 bits measured over the listed cases
    and a few drawn ones, which bounds what sums in another order differ by."""
    kind = case["kind"]
    if kind == "train" or kind == "layer":
        # a ReLU gradient is 0 or its whole cotangent: a pre-activation within rounding of zero
        # may fall on either side, and moves the gradients behind it
        return {"rel": 3e-3, "max": 0.9} if case["act"] == "relu" else {"rel": 1e-5, "max": 1e-3}
    if kind == "infer":
        return {"rel": 3e-6, "max": 1e-3}
    if kind == "softmax":  # the backward pass subtracts a row's weighted mean: it cancels
        return {"rel": 6e-5, "max": 5e-3}
    return {"rel": 1e-6, "max": 1e-4}
