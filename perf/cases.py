"""What this library is timed on: the work a program hands to it through `plast_amd`'s entry points.

Every case is one pass of one kind of work ("kind") at one size. The listed cases take the sizes of
the five benchmark configurations (bench.py) and of ordinary programs beside them; `draw` gives more
of the same kinds over their whole range: from a few hundred elements, where a call is all latency,
to the largest listed one, with odd and ragged extents among them.

Programs that launch many ops run the library in asynchronous mode (plast_hip_set_sync(0)), as these
cases do. Buffers are torch tensors on the GPU, described by `Tensor` structs; outputs and
gradients are the state's own buffers, and gradients accumulate, as the ops' contract has it.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from plast_amd import abi
from plast_amd.abi import DIM_ALL, FLOAT32, INT32, INT64, KernelParams
from plast_amd.graph import Graph
from plast_amd.runtime import backward, forward, lib

DEV = "cuda"


# ----------------------------------------------------------------------------- the cases

def listed():
    return [
        # Configuration 1: a small MLP layer's bias + ReLU, forward and backward, through the
        # scheduler's fused DAG. Latency: 1 MiB of activations.
        {"name": "bias_relu_1024x256", "kind": "bias_relu", "rows": 1024, "cols": 256, "alpha": 0.0},
        # Configuration 2: one long fused elementwise chain, exp(-relu(a * b + c)), in one launch.
        {"name": "chain_64M", "kind": "chain", "n": 1 << 26},
        # Configuration 3's chain (permute(A) + B) * C as inference runs it (one fused launch), at
        # extents that are no multiple of anything.
        {"name": "bcast_64x513x301", "kind": "bcast", "b": 64, "m": 513, "n": 301},
        # Configuration 3 as a training graph: both ops forward, then every operand's gradient.
        {"name": "bcast_train_256x512x512", "kind": "bcast_train", "b": 256, "m": 512, "n": 512},
        # Configuration 4: the four reductions of the rows of a large matrix.
        {"name": "rows_65536x4096", "kind": "rows", "rows": 65536, "cols": 4096},
        # Pooling short feature rows (mean and max), forward and backward.
        {"name": "rows_train_50000x77", "kind": "rows_train", "rows": 50000, "cols": 77},
        # Configuration 4: sum and max over the leading axis.
        {"name": "axis_4096x65536", "kind": "axis", "outer": 1, "len": 4096, "inner": 65536},
        # Configuration 5: a whole cross-entropy training step over a large vocabulary.
        {"name": "ce_step_32768x32000", "kind": "ce_step", "rows": 32768, "cols": 32000},
        # A ten-class classifier's loss over a whole data set, as the op's forward and backward.
        {"name": "ce_train_60000x10", "kind": "ce_train", "rows": 60000, "cols": 10},
        # Softmax over a thousand classes, forward and backward.
        {"name": "softmax_train_16384x1000", "kind": "softmax_train", "rows": 16384, "cols": 1000,
         "log": False},
        # A gated activation, leaky_relu(a * b + c), node by node with every gradient.
        {"name": "elementwise_train_4096x4096", "kind": "elementwise_train", "rows": 4096,
         "cols": 4096, "alpha": 0.01},
        # An optimizer step over the weights and biases of a deep MLP.
        {"name": "adam_24x1024", "kind": "optim", "rule": "adam", "layers": 24, "width": 1024},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _extent(rng, lo, hi):
    """An extent over [lo, hi], half of them as they fall and half rounded to a usual multiple."""
    n = _log_int(rng, lo, hi)
    m = rng.choice([1, 1, 1, 4, 16, 64])
    return max(lo, min(hi, n // m * m if n >= m else n))


def draw(rng):
    kind = rng.choice(["bias_relu", "chain", "bcast", "bcast_train", "rows", "rows_train", "axis",
                       "ce_step", "ce_train", "softmax_train", "elementwise_train", "optim"])
    if kind == "bias_relu":
        cols = _extent(rng, 10, 4096)
        return {"kind": kind, "rows": _extent(rng, 16, min(16384, (1 << 26) // cols)), "cols": cols,
                "alpha": rng.choice([0.0, 0.01, 0.2])}
    if kind == "chain":
        return {"kind": kind, "n": _extent(rng, 1000, 1 << 26)}
    if kind in ("bcast", "bcast_train"):
        m, n = _extent(rng, 16, 1024), _extent(rng, 16, 1024)
        return {"kind": kind, "b": _log_int(rng, 2, min(256, (1 << 26) // (m * n))), "m": m, "n": n}
    if kind in ("rows", "rows_train"):
        cols = _extent(rng, 8, 32768)
        rows = _extent(rng, 16, min(1 << 18, (1 << (28 if kind == "rows" else 26)) // cols))
        return {"kind": kind, "rows": rows, "cols": cols}
    if kind == "axis":
        n = _extent(rng, 16, 8192)
        inner = _extent(rng, 8, min(65536, (1 << 28) // n))
        outer = rng.choice([1, 1, _log_int(rng, 2, 64)])
        return {"kind": kind, "outer": max(1, min(outer, (1 << 28) // (n * inner))), "len": n,
                "inner": inner}
    if kind in ("ce_step", "ce_train"):
        cols = _extent(rng, 10, 32768)
        rows = _extent(rng, 64, min(65536, (1 << (29 if kind == "ce_step" else 28)) // cols))
        return {"kind": kind, "rows": rows, "cols": cols}
    if kind == "softmax_train":
        cols = _extent(rng, 10, 16384)
        return {"kind": kind, "rows": _extent(rng, 64, min(1 << 18, (1 << 27) // cols)), "cols": cols,
                "log": rng.random() < 0.5}
    if kind == "elementwise_train":
        cols = _extent(rng, 10, 8192)
        return {"kind": kind, "rows": _extent(rng, 16, min(1 << 16, (1 << 25) // cols)),
                "cols": cols, "alpha": rng.choice([0.0, 0.01, 0.2])}
    width = _extent(rng, 32, 2048)
    return {"kind": "optim", "rule": rng.choice(["sgd", "adam", "adamw"]),
            "layers": _log_int(rng, 2, max(2, min(48, (1 << 25) // (width * width)))),
            "width": width}


# ----------------------------------------------------------------------------- tensors

_DT = {torch.float32: FLOAT32, torch.int32: INT32, torch.int64: INT64}


class Buf:
    """A torch tensor and the `Tensor` struct that describes it (with its gradient's, if any)."""

    def __init__(self, v: torch.Tensor, grad: "torch.Tensor | None" = None):
        self.v, self.g = v, grad
        self.gt = None
        if grad is not None:
            self.gt = abi.make_tensor(grad.data_ptr(), grad.shape, grad.stride(), FLOAT32)
        self.t = abi.make_tensor(v.data_ptr(), v.shape, v.stride(), _DT[v.dtype],
                                 requires_grad=grad is not None, grad=self.gt)


def _ready():
    # the library's stream is its own: the inputs torch has made are waited for before the first call
    lib().plast_hip_set_sync(0)
    torch.cuda.synchronize()


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, sd=1.0):
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    return x if sd == 1.0 else x.mul_(sd)


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float32).mul_(hi - lo).add_(lo)


def _empty(shape, dtype=torch.float32):
    return torch.empty(shape, device=DEV, dtype=dtype)


def _zeros(shape):
    return torch.zeros(shape, device=DEV, dtype=torch.float32)


def _leaf(v, grad=True):
    return Buf(v, torch.zeros_like(v) if grad else None)


def _mid(shape):
    """An op's output that carries a gradient."""
    return Buf(_empty(shape), _zeros(shape))


# ----------------------------------------------------------------------------- inputs

def _inputs(case, seed):
    """The input values of a case, from the seed alone (shared by prepare and exact)."""
    g, k = _gen(seed), case["kind"]
    if k == "bias_relu":
        s = (case["rows"], case["cols"])
        return {"x": _uniform(g, s, -1, 1), "b": _uniform(g, s[1:], -1, 1), "dy": _normal(g, s)}
    if k == "chain":
        return {n: _normal(g, (case["n"],)) for n in "abc"}
    if k in ("bcast", "bcast_train"):
        b, m, n = case["b"], case["m"], case["n"]
        d = {"a": _normal(g, (b, n, m)), "b": _uniform(g, (1, m, 1), 0.5, 1.5),
             "c": _uniform(g, (b, 1, n), 0.5, 1.5)}
        if k == "bcast_train":
            d["dy"] = _normal(g, (b, m, n))
        return d
    if k == "rows":
        return {"x": _normal(g, (case["rows"], case["cols"]))}
    if k == "rows_train":
        return {"x": _normal(g, (case["rows"], case["cols"])),
                "dmean": _normal(g, (case["rows"],)), "dmax": _normal(g, (case["rows"],))}
    if k == "axis":
        return {"x": _normal(g, (case["outer"], case["len"], case["inner"]))}
    if k in ("ce_step", "ce_train"):
        n, c = case["rows"], case["cols"]
        return {"x": _normal(g, (n, c), 2.0),
                "y": torch.randint(0, c, (n,), generator=g, device=DEV, dtype=torch.int32),
                "dl": torch.full((n,), 1.0 / n, device=DEV, dtype=torch.float32)}
    if k == "softmax_train":
        s = (case["rows"], case["cols"])
        return {"x": _normal(g, s, 2.0), "dy": _normal(g, s)}
    if k == "elementwise_train":
        s = (case["rows"], case["cols"])
        return {n: _normal(g, s) for n in ("a", "b", "c", "dy")}
    n = sum(_slots(case)[1])
    return {"p": _normal(g, (n,), 0.05), "g": _normal(g, (n,), 0.01), "m": _normal(g, (n,), 0.01),
            "v": _uniform(g, (n,), 1e-6, 1e-4)}


def _slots(case):
    """Shapes of the parameters (each layer's weight and bias) and the floats each one's slot of a
    flat buffer takes: slots start on 256-byte boundaries, as separate allocations do."""
    w = case["width"]
    shapes = [s for _ in range(case["layers"]) for s in ((w, w), (w,))]
    return shapes, [-(-math.prod(s) // 64) * 64 for s in shapes]


def _split(case, flat):
    """The parameters inside a flat buffer."""
    out, off = [], 0
    for shape, slot in zip(*_slots(case)):
        out.append(flat[off:off + math.prod(shape)].view(shape))
        off += slot
    return out


LR, B1, B2, EPS, DECAY, T0 = 1e-3, 0.9, 0.999, 1e-8, 0.01, 9  # the optimizers, nine steps in


# ----------------------------------------------------------------------------- prepare and run

def prepare(case, seed):
    d, k = _inputs(case, seed), case["kind"]
    s = {"kind": k, "case": dict(case)}
    if k == "bias_relu":
        shape = d["x"].shape
        x, b = _leaf(d["x"]), _leaf(d["b"])
        mid, y = _mid(shape), Buf(_empty(shape), d["dy"])
        g = Graph()
        g.node("add", [x, b], mid)
        g.node("leaky_relu", [mid], y, KernelParams(0, 0, case["alpha"]))
        g.build(y, fuse=True)
        s.update(g=g, out={"y": y.v, "dx": x.g, "db": b.g}, keep=(x, b, mid, y))
    elif k == "chain":
        a, b, c = (Buf(d[n]) for n in "abc")
        t = [Buf(_empty((case["n"],))) for _ in range(4)]  # the chain's own, not written once fused
        y = Buf(_empty((case["n"],)))
        g = Graph()
        g.node("mul", [a, b], t[0])
        g.node("add", [t[0], c], t[1])
        g.node("leaky_relu", [t[1]], t[2], KernelParams(0, 0, 0.0))
        g.node("neg", [t[2]], t[3])
        g.node("exp", [t[3]], y)
        if g.build(y, fuse=True) != 1:
            raise RuntimeError("the chain was not fused")
        s.update(g=g, out=y.v, keep=(a, b, c, t, y))
    elif k == "bcast":
        shape = (case["b"], case["m"], case["n"])
        a, b, c = Buf(d["a"].transpose(1, 2)), Buf(d["b"]), Buf(d["c"])
        t, y = Buf(_empty(shape)), Buf(_empty(shape))
        g = Graph()
        g.node("add", [a, b], t)
        g.node("mul", [t, c], y)
        if g.build(y, fuse=True) != 1:
            raise RuntimeError("the chain was not fused")
        s.update(g=g, out=y.v, keep=(a, b, c, t, y))
    elif k == "bcast_train":
        shape = (case["b"], case["m"], case["n"])
        a = Buf(d["a"].transpose(1, 2), torch.zeros_like(d["a"]).transpose(1, 2))
        b, c = _leaf(d["b"]), _leaf(d["c"])
        t, y = _mid(shape), Buf(_empty(shape), d["dy"])
        g = Graph()
        g.node("add", [a, b], t)
        g.node("mul", [t, c], y)
        g.build(y)
        s.update(g=g, out={"y": y.v, "da": a.g, "db": b.g, "dc": c.g}, keep=(a, b, c, t, y))
    elif k == "rows":
        x, n = Buf(d["x"]), case["rows"]
        s.update(x=x, sum=Buf(_empty((n,))), mean=Buf(_empty((n,))), max=Buf(_empty((n,))),
                 argmax=Buf(_empty((n,), torch.int64)))
    elif k == "rows_train":
        n = case["rows"]
        x = _leaf(d["x"])
        s.update(x=x, mean=Buf(_empty((n,)), d["dmean"]), max=Buf(_empty((n,)), d["dmax"]))
    elif k == "axis":
        x, o = Buf(d["x"]), (case["outer"], case["inner"])
        s.update(x=x, sum=Buf(_empty(o)), max=Buf(_empty(o)))
    elif k == "ce_step":
        n, c = case["rows"], case["cols"]
        s.update(d=d, n=n, c=c, out={"stats": _empty((n, 2)), "loss": _empty((n,)),
                                     "dx": _empty((n, c)), "db": _empty((c,)), "mean": _empty((1,))})
    elif k == "ce_train":
        n = case["rows"]
        s.update(x=_leaf(d["x"]), y=Buf(d["y"]), stats=Buf(_empty((n, 2))),
                 loss=Buf(_empty((n,)), d["dl"]))
    elif k == "softmax_train":
        s.update(x=_leaf(d["x"]), y=Buf(_empty(d["x"].shape), d["dy"]),
                 op="log_softmax" if case["log"] else "softmax")
    elif k == "elementwise_train":
        shape = d["a"].shape
        a, b, c = (_leaf(d[n]) for n in "abc")
        m, r, y = _mid(shape), _mid(shape), Buf(_empty(shape), d["dy"])
        s.update(a=a, b=b, c=c, m=m, r=r, y=y)
    else:
        ps = [Buf(p, g) for p, g in zip(_split(case, d["p"]), _split(case, d["g"]))]
        arr = (abi.TensorP * len(ps))(*[C.pointer(p.t) for p in ps])
        s.update(ps=ps, arr=arr, n=len(ps), out={n: d[n] for n in "pmv"}, keep=[d["g"]])
        if case["rule"] == "sgd":
            s["out"] = {"p": d["p"]}
            s["opt"] = abi.SGD(LR)
        else:
            ms, vs = ([Buf(x) for x in _split(case, d[n])] for n in "mv")
            ma = (abi.TensorP * len(ms))(*[C.pointer(x.t) for x in ms])
            va = (abi.TensorP * len(vs))(*[C.pointer(x.t) for x in vs])
            o = abi.Adam() if case["rule"] == "adam" else abi.AdamW()
            o.lr, o.beta1, o.beta2, o.epsilon, o.t = LR, B1, B2, EPS, T0
            if case["rule"] == "adamw":
                o.weight_decay = DECAY
            o.m, o.v = C.cast(ma, abi.TensorPP), C.cast(va, abi.TensorPP)
            s["opt"] = o
            s["keep"] += [ms, vs, ma, va]
    _ready()
    return s


_ROW = KernelParams(1, 0, 0.0)


def run(s):
    k = s["kind"]
    if k in ("chain", "bcast"):
        s["g"].forward()
        return s["out"]
    if k in ("bias_relu", "bcast_train"):
        s["g"].forward()
        s["g"].backward()
        return s["out"]
    if k == "rows":
        for op in ("sum", "mean", "max", "argmax"):
            forward(op, [s["x"].t], s[op].t, _ROW)
        return {op: s[op].v for op in ("sum", "mean", "max", "argmax")}
    if k == "rows_train":
        for op in ("mean", "max"):
            forward(op, [s["x"].t], s[op].t, _ROW)
        for op in ("max", "mean"):
            backward(op, [s["x"].t], s[op].t, _ROW)
        return {"mean": s["mean"].v, "max": s["max"].v, "dx": s["x"].g}
    if k == "axis":
        for op in ("sum", "max"):
            forward(op, [s["x"].t], s[op].t, _ROW)
        return {"sum": s["sum"].v, "max": s["max"].v}
    if k == "ce_step":
        d, o = s["d"], s["out"]
        L = lib()
        L.softmax_cross_entropy_step_hip(
            d["x"].data_ptr(), d["y"].data_ptr(), d["dl"].data_ptr(), o["stats"].data_ptr(),
            o["loss"].data_ptr(), o["dx"].data_ptr(), o["db"].data_ptr(), o["mean"].data_ptr(),
            s["n"], s["c"])
        L.check("cross-entropy step")
        return o
    if k == "ce_train":
        ins = [s["x"].t, s["y"].t, s["stats"].t]
        forward("softmax_cross_entropy", ins, s["loss"].t)
        backward("softmax_cross_entropy", ins, s["loss"].t)
        return {"loss": s["loss"].v, "stats": s["stats"].v, "dx": s["x"].g}
    if k == "softmax_train":
        forward(s["op"], [s["x"].t], s["y"].t, _ROW)
        backward(s["op"], [s["x"].t], s["y"].t, _ROW)
        return {"y": s["y"].v, "dx": s["x"].g}
    if k == "elementwise_train":
        a, b, c, m, r, y = (s[n].t for n in ("a", "b", "c", "m", "r", "y"))
        p = KernelParams(0, 0, s["case"]["alpha"])
        forward("mul", [a, b], m)
        forward("add", [m, c], r)
        forward("leaky_relu", [r], y, p)
        backward("leaky_relu", [r], y, p)
        backward("add", [m, c], r)
        backward("mul", [a, b], m)
        return {"y": s["y"].v, "da": s["a"].g, "db": s["b"].g, "dc": s["c"].g}
    L = lib()
    getattr(L, s["case"]["rule"] + "_step_hip")(C.byref(s["opt"]), s["arr"], s["n"])
    L.check("optimizer step")
    return s["out"]


# ----------------------------------------------------------------------------- work

def work(case):
    """Bytes and operations of one pass. Each call of a pass reads its inputs once and writes its
    outputs once (an accumulated gradient is both); broadcast operands count their own elements."""
    k = case["kind"]
    if k == "bias_relu":  # forward x -> y; backward dy, y, dx -> dx
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * (2 * n + 4 * n + 3 * case["cols"]), "flops": 5 * n}
    if k == "chain":
        return {"bytes": 16 * case["n"], "flops": 5 * case["n"]}
    if k in ("bcast", "bcast_train"):
        n = case["b"] * case["m"] * case["n"]
        small = case["m"] + case["b"] * case["n"]
        if k == "bcast":
            return {"bytes": 4 * (2 * n + small), "flops": 2 * n}
        # add a -> t; mul t -> y; mul's backward dy, t, dt -> dt; add's backward dt, da -> da
        return {"bytes": 4 * (2 * n + 2 * n + 4 * n + 3 * n + 5 * small), "flops": 7 * n}
    if k == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * (4 * n + 5 * case["rows"]), "flops": 4 * n}
    if k == "rows_train":  # two forwards x; max's backward x, dx -> dx; mean's dx -> dx
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * (2 * n + 3 * n + 2 * n + 5 * case["rows"]), "flops": 5 * n}
    if k == "axis":
        n = case["outer"] * case["len"] * case["inner"]
        return {"bytes": 4 * (2 * n + 2 * case["outer"] * case["inner"]), "flops": 2 * n}
    if k == "ce_step":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n + 24 * case["rows"] + 4 * case["cols"] + 4, "flops": 9 * n}
    if k == "ce_train":  # forward x; backward x, dx -> dx
        n = case["rows"] * case["cols"]
        return {"bytes": 16 * n + 32 * case["rows"], "flops": 9 * n}
    if k == "softmax_train":  # forward x -> y; backward y, dy, dx -> dx
        n = case["rows"] * case["cols"]
        return {"bytes": 24 * n, "flops": 9 * n}
    if k == "elementwise_train":
        # mul a, b -> m; add m, c -> r; leaky r -> y; its backward dy, r, dr -> dr; add's backward
        # dr, dm -> dm, dc -> dc; mul's backward dm, a, b, da -> da, db -> db
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * 24 * n, "flops": 10 * n}
    n = case["layers"] * case["width"] * (case["width"] + 1)
    if case["rule"] == "sgd":
        return {"bytes": 12 * n, "flops": 2 * n}
    return {"bytes": 28 * n, "flops": 12 * n}


# ----------------------------------------------------------------------------- tolerance

def tolerance(case):
    """Relative 2-norm errors another correct fp32 implementation would show: sums in another order
    and exponentials of another rounding; indices are exact."""
    k = case["kind"]
    if k in ("chain", "bcast", "optim"):  # elementwise: a few roundings each
        return {"rel": 1e-6, "max": 2e-5}
    if k == "bcast_train":  # b's gradient: up to 2^18 terms an element, 6e-6 off when summed in series
        return {"rel": 3e-5, "max": 1e-3}
    return {"rel": 4e-6, "max": 1e-3, "differ": 0.0}


# ----------------------------------------------------------------------------- exact

def exact(case, seed):
    d, k = _inputs(case, seed), case["kind"]
    if k == "optim":
        return _exact_optim(case, d)
    if k in ("ce_step", "ce_train"):
        return _exact_ce(case, d)
    if k == "bias_relu":
        r = d["x"].double() + d["b"].double()
        m = torch.where(r > 0, 1.0, float(torch.tensor(case["alpha"], dtype=torch.float32)))
        dx = d["dy"].double() * m
        return {"y": r * m, "dx": dx, "db": dx.sum(0)}
    if k == "chain":
        y = d["a"].double().mul_(d["b"].double()).add_(d["c"].double())
        return y.clamp_(min=0).neg_().exp_()
    if k == "bcast":
        return (d["a"].double().transpose(1, 2) + d["b"].double()).mul_(d["c"].double())
    if k == "bcast_train":
        t = d["a"].double().transpose(1, 2) + d["b"].double()
        c, dy = d["c"].double(), d["dy"].double()
        dt = dy * c
        return {"y": t * c, "da": dt, "db": dt.sum((0, 2), keepdim=True),
                "dc": dy.mul_(t).sum(1, keepdim=True)}
    if k == "rows":
        x = d["x"]
        s = x.sum(1, dtype=torch.float64)
        return {"sum": s, "mean": s / x.shape[1], "max": x.amax(1).double(), "argmax": None}
    if k == "rows_train":
        x = d["x"]
        mx = x.amax(1, keepdim=True)
        tie = (x == mx).double()
        dx = tie * (d["dmax"].double()[:, None] / tie.sum(1, keepdim=True))
        dx += d["dmean"].double()[:, None] / x.shape[1]
        return {"mean": x.mean(1, dtype=torch.float64), "max": mx[:, 0].double(), "dx": dx}
    if k == "axis":
        return {"sum": d["x"].sum(1, dtype=torch.float64), "max": d["x"].amax(1).double()}
    if k == "softmax_train":
        x, dy = d["x"].double(), d["dy"].double()
        if case["log"]:
            y = torch.log_softmax(x, 1)
            return {"y": y, "dx": dy - y.exp() * dy.sum(1, keepdim=True)}
        y = torch.softmax(x, 1)
        return {"y": y, "dx": y * (dy - (dy * y).sum(1, keepdim=True))}
    a, b, c, dy = (d[n].double() for n in ("a", "b", "c", "dy"))
    r = a * b + c
    m = torch.where(r > 0, 1.0, float(torch.tensor(case["alpha"], dtype=torch.float32)))
    g = dy * m
    return {"y": r * m, "da": g * b, "db": g * a, "dc": g}


def _exact_ce(case, d):
    x, n, c = d["x"], case["rows"], case["cols"]
    mx = x.amax(1).double()
    lse, xy = (torch.empty(n, device=DEV, dtype=torch.float64) for _ in range(2))
    dx = torch.empty((n, c), device=DEV, dtype=torch.float64)
    g = d["dl"].double()
    for r0 in range(0, n, 4096):  # a few rows at a time: the whole is 8 GiB and more in 64 bits
        r = slice(r0, min(n, r0 + 4096))
        t = x[r].double().sub_(mx[r, None])
        y = d["y"][r].long()[:, None]
        xy[r] = t.gather(1, y)[:, 0]
        lse[r] = t.exp().sum(1).log_()
        t.sub_(lse[r, None]).exp_()
        t.scatter_add_(1, y, torch.full_like(y, -1.0, dtype=torch.float64))
        dx[r] = t.mul_(g[r, None])
    out = {"loss": lse - xy, "stats": torch.stack([mx, lse], 1), "dx": dx}
    if case["kind"] == "ce_step":
        out.update(db=dx.sum(0), mean=(lse - xy).mean().reshape(1))
    return out


def _exact_optim(case, d):
    def f32(v):
        return float(torch.tensor(v, dtype=torch.float32))

    lr, b1, b2, eps = f32(LR), f32(B1), f32(B2), f32(EPS)
    out = {n: d[n].double() for n in (("p",) if case["rule"] == "sgd" else ("p", "m", "v"))}
    flat = {n: _split(case, out[n]) for n in out}
    for i, g in enumerate(_split(case, d["g"])):
        g, p = g.double(), flat["p"][i]
        if case["rule"] == "sgd":
            p.sub_(lr * g)
            continue
        m, v = flat["m"][i], flat["v"][i]
        if case["rule"] == "adamw":
            p.sub_(lr * f32(DECAY) * p)
        m.mul_(b1).add_((1 - b1) * g)
        v.mul_(b2).add_((1 - b2) * g * g)
        step = lr * math.sqrt(1 - b2 ** (T0 + 1)) / (1 - b1 ** (T0 + 1))
        p.sub_(step * m / (v.sqrt() + eps))
    return out
