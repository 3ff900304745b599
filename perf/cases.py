"""Work that a program on this backend does, as cases for timing and comparing.

A case is one compiled routine: what ``Train.to_routine`` (or a forward-only caller) hands over, compiled
once per program, linked against a context that holds the inputs, and run.  One pass is one
``Routine.run`` -- for the training routines forward, backward and optimiser update together, the next
batch selected by the static index.  The families:

  moons        the half-moons MLP with SGD and momentum: the smallest routine anyone trains (a launch and
               its latency are all of it)
  char_mlp     the character-level MLP language model with Adam: small, fp32, many small parameters
  transformer  the decoder-only training step: bf16 values with fp32 gradients, or fp32 throughout; in
               the routine form of single-reader inlining or of the visit rule
  dense        ``b|i->o`` with both gradients, or forward only (a serving batch), fp32 and bf16 operands
  attention    batched soft-max attention, forward with or without backward
  conv         a convolution layer, forward with both gradients (windows ``stride * o + k``)

Results stay in device memory, where the framework keeps them: ``run`` returns a dict that copies a
node to the host when its entry is read, as ``Context.get_values`` does for any program.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ocannl_amd import backend as B
from ocannl_amd import llir as L
from ocannl_amd import workloads as W


def listed():
    return [
        # the first thing a new user trains; one tiny kernel, so latency is everything
        dict(name="moons_step", family="moons", batch=20, hidden=16),
        # the names-model of the reference's training tests
        dict(name="char_mlp_step", family="char_mlp", batch=32, vocab=27, context=3, embed=10, hidden=200),
        # a transformer small enough to debug with: a few dozen launches of very little work
        dict(name="transformer_small_f32", family="transformer", batch=2, seq=16, d_model=32, heads=2, d_ff=64, layers=2, vocab=64,
             prec="single", inline="reads"),
        # the benchmark training step (configuration 4)
        dict(name="transformer_step", family="transformer", batch=32, seq=256, d_model=512, heads=8, d_ff=2048, layers=4, vocab=4096,
             prec="bfloat16", inline="reads"),
        # the same model as somebody sizes it for their own data: a vocabulary and a sequence length that are
        # not multiples of anything, in the visit-rule form
        dict(name="transformer_odd", family="transformer", batch=6, seq=99, d_model=320, heads=5, d_ff=1280, layers=2, vocab=1003,
             prec="bfloat16", inline="visits"),
        # configuration 3 in its two precisions: the largest contractions
        dict(name="dense_bf16", family="dense", b=8192, i=4096, o=4096, prec="bfloat16", which="all"),
        dict(name="dense_f32", family="dense", b=8192, i=4096, o=4096, prec="single", which="all"),
        # a layer with odd extents on every axis
        dict(name="dense_bf16_odd", family="dense", b=1777, i=1001, o=771, prec="bfloat16", which="all"),
        # a layer applied to one serving batch: the weights are all there is to read
        dict(name="dense_serve", family="dense", b=64, i=4096, o=4096, prec="bfloat16", which="fwd"),
        # configuration 5, forward and backward
        dict(name="attention", family="attention", b=16, h=16, q=1024, k=1024, d=64, prec="bfloat16", backward=True),
        # attention over patches and a class token: forward only, odd length
        dict(name="attention_fwd_odd", family="attention", b=8, h=12, q=197, k=197, d=64, prec="bfloat16", backward=False),
        # a layer of an image classifier
        dict(name="conv_layer", family="conv", b=64, oh=32, ow=32, ic=32, oc=64, ksz=3, stride=1, prec="single"),
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm: odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(("moons", "char_mlp", "transformer", "transformer", "dense", "dense", "dense", "attention", "attention", "conv"))
    prec = rng.choice(("bfloat16", "single"))
    if family == "moons":
        return dict(family=family, batch=_between(rng, 5, 128), hidden=_between(rng, 8, 64))
    if family == "char_mlp":
        return dict(family=family, batch=_between(rng, 8, 128), vocab=_between(rng, 20, 128), context=rng.randint(2, 6),
                    embed=_between(rng, 6, 32), hidden=_between(rng, 48, 512))
    if family == "transformer":
        heads = rng.randint(1, 8)
        d_model = heads * rng.choice((16, 32, 64))
        return dict(family=family, batch=_between(rng, 2, 32), seq=_between(rng, 16, 256), d_model=d_model, heads=heads,
                    d_ff=d_model * rng.choice((2, 4)), layers=rng.randint(1, 3), vocab=_between(rng, 64, 4096), prec=prec,
                    inline=rng.choice(("reads", "visits")))
    if family == "dense":
        # layer widths are multiples of eight about half the time, batches are what they are
        width = lambda hi: (lambda n: n if rng.random() < 0.5 else max(64, n // 8 * 8))(_between(rng, 64, hi))
        if rng.random() < 0.3:
            return dict(family=family, b=_between(rng, 16, 256), i=width(4096), o=width(4096), prec=prec, which="fwd")
        return dict(family=family, b=_between(rng, 128, 8192), i=width(4096), o=width(4096), prec=prec, which="all")
    if family == "attention":
        q = _between(rng, 32, 1024)
        return dict(family=family, b=_between(rng, 1, 8), h=rng.randint(2, 16), q=q, k=q, d=rng.choice((32, 64)), prec=prec,
                    backward=rng.random() < 0.5)
    return dict(family=family, b=_between(rng, 8, 64), oh=_between(rng, 8, 32), ow=_between(rng, 8, 32), ic=_between(rng, 3, 32),
                oc=_between(rng, 8, 64), ksz=rng.choice((3, 5)), stride=rng.choice((1, 1, 2)), prec=prec)


# ---- routines ------------------------------------------------------------------------------------

def _conv_layer(b, oh, ow, ic, oc, ksz, stride, prec):
    """``y[b,oh,ow,oc] = sum x[b, stride*oh+kh, stride*ow+kw, ic] * w[oc,kh,kw,ic]`` and the gradients of x and
    w from a supplied gradient of y (lib/nn_blocks.ml:418-428; gradients in single precision)."""
    L.reset_symbols(0)
    ih, iw = stride * (oh - 1) + ksz, stride * (ow - 1) + ksz
    nodes = dict(x=L.Node(1, "x", prec, (b, ih, iw, ic)), w=L.Node(2, "w", prec, (oc, ksz, ksz, ic)), y=L.Node(3, "y", prec, (b, oh, ow, oc)),
                 dy=L.Node(4, "y_grad", prec, (b, oh, ow, oc)), dx=L.Node(5, "x_grad", "single", (b, ih, iw, ic)),
                 dw=L.Node(6, "w_grad", "single", (oc, ksz, ksz, ic)))

    def nest(lhs, p, q):
        s = [L.fresh_symbol() for _ in range(7)]
        bb, o1, o2, c, k1, k2, i = s
        at = dict(x=(L.It(bb), L.Affine(((stride, o1), (1, k1)), 0), L.Affine(((stride, o2), (1, k2)), 0), L.It(i)),
                  y=(L.It(bb), L.It(o1), L.It(o2), L.It(c)), w=(L.It(c), L.It(k1), L.It(k2), L.It(i)))
        get = lambda n: L.Get(nodes[n], at[n.lstrip("d")])
        body = [L.Set(nodes[lhs], at[lhs.lstrip("d")], L.Ternop("fma", get(p), get(q), get(lhs)))]
        for sym, ext in reversed(list(zip(s, (b, oh, ow, oc, ksz, ksz, ic)))):
            body = [L.For(sym, 0, ext - 1, body)]
        return [L.ZeroOut(nodes[lhs])] + body

    return L.Routine("conv_layer", nest("y", "x", "w") + nest("dx", "dy", "w") + nest("dw", "dy", "x")), nodes


class _Program:
    """What a program keeps for all its inputs: the routine, its compiled code, and where its tensors are."""

    def __init__(self, case):
        self.statics, f = [], case["family"]
        if f == "conv":
            self.routine, nodes = _conv_layer(**{k: case[k] for k in ("b", "oh", "ow", "ic", "oc", "ksz", "stride", "prec")})
            self.outputs = {n: [nodes[n]] for n in ("y", "dx", "dw")}
        else:
            w = _workload(case, 0)
            self.routine, nodes = w.routine, w.nodes
            self.statics = list(w.statics.values())
            if f == "dense":
                self.outputs = {n.ident.rsplit("_", 1)[0]: [n] for n in w.outputs}
            elif f == "attention":
                self.outputs = {n: [nodes[n]] for n in (("out", "dq", "dk", "dv") if case["backward"] else ("out",))}
            elif f == "transformer":
                # the parameters layer by layer, and the gradients of the last layer and of the output projection.
                # (Gradients further back pass through layer norms that subtract the SUM over the axis
                # (lib/nn_blocks.ml:251-258): small differences of large values, in which two correct orders of
                # summation lie tens of percent apart in bf16 and 3e-3 in fp32, so they say nothing.)
                self.outputs = {"loss": [nodes["loss"]], "logits": [nodes["logits"]]}
                last = f"l{case['layers'] - 1}"
                for p in w.params:
                    tail = p.label.rsplit("_", 1)[1]
                    group = tail if tail[0] == "l" and tail[1:].isdigit() else p.label
                    self.outputs.setdefault(group, []).append(p.value)
                    if group in (last, "w_out") and p.grad.mode == "ctx":
                        self.outputs.setdefault(group + "_grad", []).append(p.grad)
            else:
                self.outputs = {n: [v] for n, v in nodes.items() if n not in ("data", "classes")}
            w.init.clear()
        self.outputs = {k: [n for n in v if n.mode == "ctx"] for k, v in self.outputs.items()}
        self.outputs = {k: v for k, v in self.outputs.items() if v}
        self.code = B.compile(self.routine)


def _workload(case, seed):
    c = {k: v for k, v in case.items() if k not in ("name", "family")}
    if case["family"] == "moons":
        return W.moons_mlp(seed=seed, **c)
    if case["family"] == "char_mlp":
        return W.char_mlp(seed=seed, **c)
    if case["family"] == "transformer":
        return W.transformer(seed=seed, grad_prec="single", **dict(c, inline=True if c["inline"] == "reads" else "visits"))
    if case["family"] == "dense":
        which = ("fwd", "dx", "dw") if c.pop("which") == "all" else ("fwd",)
        return W.dense_contraction(out_prec="single", which=which, seed=seed, **c)
    return W.attention(grad_prec="single", seed=seed, **c)


_programs: dict = {}


def _program(case):
    """Compiled once per process, as a program compiles its routine once."""
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _programs:
        _programs[key] = _Program(case)
    return _programs[key]


# ---- inputs --------------------------------------------------------------------------------------

def _host(t, prec):
    t = t.to({"single": torch.float32, "bfloat16": torch.bfloat16}[prec]).contiguous().cpu()
    return t.numpy() if prec == "single" else t.view(torch.int16).numpy().view(np.uint16)


def _inputs(case, program, seed):
    """Node id -> values, with the distributions of the benchmark configurations."""
    if case["family"] in ("moons", "char_mlp"):
        return _workload(case, seed).init
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(dev).manual_seed(seed)
    uniform = lambda dims: torch.rand(dims, generator=gen, device=dev) * 2 - 1
    init = {}
    for n in program.routine.param_nodes():
        name = n.ident.rsplit("_", 1)[0] if n.ident.rsplit("_", 1)[-1].isdigit() else n.ident
        if case["family"] == "attention":
            if name in ("q", "k", "v", "attn_out_grad"):
                init[n.id] = _host(torch.randn(n.dims, generator=gen, device=dev), n.prec)
        elif case["family"] in ("dense", "conv"):
            if name in ("x", "w", "dy", "y_grad"):
                init[n.id] = _host(uniform(n.dims), n.prec)
        elif name in ("input_batch", "target_batch"):
            toks = torch.randint(0, n.dims[-1], n.dims[:-1], generator=gen, device=dev)
            hot = torch.zeros(n.dims, device=dev, dtype=torch.bfloat16 if n.prec == "bfloat16" else torch.float32)
            init[n.id] = _host(hot.scatter_(-1, toks.unsqueeze(-1), 1.0), n.prec)
        elif name == "mask":
            init[n.id] = np.tril(np.ones(n.dims, np.float32))
        elif name == "learning_rate":
            init[n.id] = np.array([0.01], np.float32)
        elif getattr(n, "_is_param", False):
            if name.startswith("gamma"):
                init[n.id] = _host(torch.ones(n.dims, device=dev), n.prec)
            elif name.startswith(("beta", "b_")):
                init[n.id] = _host(torch.zeros(n.dims, device=dev), n.prec)
            else:
                fan_in = {"w_o": n.dims[-1] * n.dims[-2]}.get(name[:3], n.dims[-1]) if len(n.dims) > 1 else n.dims[0]
                init[n.id] = _host(uniform(n.dims) * math.sqrt(3.0 / fan_in), n.prec)
    return init


class _Results(dict):
    """Name -> values as float32, copied from the device when read."""

    def __init__(self, ctx, nodes):
        super().__init__(nodes)
        self._ctx = ctx

    def __getitem__(self, name):
        nodes = super().__getitem__(name)
        vals = [self._ctx.get_values(n) for n in nodes]
        vals = [W.from_bf16_bits(v) if n.prec == "bfloat16" else v for n, v in zip(nodes, vals)]
        return vals[0] if len(vals) == 1 else np.concatenate([v.ravel() for v in vals])


class _Context(B.Context):
    """A context whose pools go when nothing refers to it any more."""

    def __del__(self):
        if self.pools:
            self.free()


class _State:
    def __init__(self, program, init):
        ctx = _Context()
        nodes = program.routine.param_nodes()
        ctx.allocate(nodes)
        for n in nodes:
            if n.id in init:
                ctx.set_values(n, init[n.id])
        self.routine = ctx.link(program.code)
        self.results = _Results(ctx, program.outputs)
        self.statics, self.passes = program.statics, 0


def prepare(case, seed):
    program = _program(case)
    return _State(program, _inputs(case, program, seed))


def run(state):
    for s in state.statics:   # the next batch
        state.routine.set_static(s.sym, state.passes % s.range)
    state.passes += 1
    state.routine.run()
    return state.results


# ---- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    """Flops of the contractions; bytes of the context tensors, which the routine has to leave in memory: each
    once, the updated ones twice."""
    c = dict(case)
    vb = 2 if c.get("prec") == "bfloat16" else 4
    if c["family"] == "moons":
        params = 2 * c["hidden"] + c["hidden"] ** 2 + 3 * c["hidden"]
        return {"bytes": 16 * params + 12 * c["batch"], "flops": 6 * c["batch"] * params}
    if c["family"] == "char_mlp":
        params = c["embed"] * c["vocab"] + c["hidden"] * (c["context"] * c["embed"] + 1) + c["vocab"] * (c["hidden"] + 1)
        return {"bytes": 24 * params + 4 * c["batch"] * (c["context"] + c["vocab"]),
                "flops": 6 * c["batch"] * (c["hidden"] * c["context"] * c["embed"] + c["vocab"] * c["hidden"])}
    if c["family"] == "dense":
        x, w, y = c["b"] * c["i"], c["i"] * c["o"], c["b"] * c["o"]
        if c["which"] == "fwd":
            return {"bytes": (x + w) * vb + y * 4, "flops": 2 * x * c["o"]}
        return {"bytes": (x + w + y) * vb + y * 4 + (x + w) * 8, "flops": 6 * x * c["o"]}
    if c["family"] == "conv":
        ih, iw = c["stride"] * (c["oh"] - 1) + c["ksz"], c["stride"] * (c["ow"] - 1) + c["ksz"]
        x, y, w = c["b"] * ih * iw * c["ic"], c["b"] * c["oh"] * c["ow"] * c["oc"], c["oc"] * c["ksz"] ** 2 * c["ic"]
        return {"bytes": (x + 2 * y + w) * vb + (x + w) * 4, "flops": 6 * y * c["ksz"] ** 2 * c["ic"]}
    if c["family"] == "attention":
        qs, s = c["b"] * c["q"] * c["h"] * c["d"], c["b"] * c["h"] * c["q"] * c["k"]
        fwd = {"bytes": 4 * qs * vb + 3 * s * vb, "flops": 4 * s * c["d"]}
        return {"bytes": fwd["bytes"] + 16 * qs + 20 * s, "flops": 3 * fwd["flops"]} if c["backward"] else fwd
    rows, d, ff, v, n = c["batch"] * c["seq"], c["d_model"], c["d_ff"], c["vocab"], c["layers"]
    s = c["batch"] * c["heads"] * c["seq"] ** 2
    weights = n * (4 * d * d + 2 * d * ff + 4 * d + ff) + 2 * d * v + d * c["seq"]
    visits = c["inline"] == "visits"
    per_layer = (s * (3 * vb + (16 if visits else 24)) + rows * ff * ((1 if visits else 2) * vb + (8 if visits else 12)) +
                 rows * d * ((8 if visits else 12) * vb + (60 if visits else 84)))
    return {"bytes": weights * (2 * vb + 4) + n * per_layer + rows * v * (3 * vb + (12 if visits else 16)),
            "flops": 6 * rows * (n * (4 * d * d + 2 * d * ff) + d * v) + 4 * rows * d * v + 12 * n * s * d // c["heads"]}


def tolerance(case):
    """fp32 sums in another order, or bf16 values rounded from sums in another order."""
    if case["family"] == "transformer":
        return {"rel": 2e-2, "max": 0.9} if case["prec"] == "bfloat16" else {"rel": 1e-4, "max": 1e-2}
    if case["family"] in ("moons", "char_mlp"):
        return {"rel": 1e-4, "max": 1e-2}
    if case["family"] == "attention" and case["prec"] == "bfloat16":
        return {"rel": 1e-2, "max": 0.5}
    if case["family"] == "conv" and case["prec"] == "bfloat16":
        return {"rel": 5e-3, "max": 0.2}
    return {"rel": 2e-5, "max": 1e-3}
