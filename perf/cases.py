"""The work that programs give this library, as cases to time and compare.

A case is one pass of a program that keeps a model's projections on the GPU:
a single projection of fp32 activations, an FFN, a layer (or two) of a question
or of a prompt, several questions' stacked rows, or a weight load.  Shapes are
the 2048-hidden model's (bench.py: 2048 -> 8224 Gated DeltaNet in, 2048 ->
2048/512/512 q/k/v, 2048 -> 2048 out, the 2048 <-> 6144 SwiGLU FFN) and generic
odd ones.  Activations are N(0, 1) with 1% of the channels scaled x20, weights
N(0, 0.02^2), adapters rank 16 as the checkpoints carry them.

Every result is compared exactly: the library's contract is the reference's own
bits (one order of every sum, each operation rounded once), so a change of
rounding anywhere is an error.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "decider-engine_amd"))
import dq8  # noqa: E402

HIDDEN, INTER, GDN_IN, KV = 2048, 6144, 8224, 512
LORA_SCALE = 0.5
GDN = (("in", HIDDEN, GDN_IN),)  # the projections of a layer's own input
GQA = (("q", HIDDEN, HIDDEN), ("k", HIDDEN, KV), ("v", HIDDEN, KV))


def listed():
    return [
        # One token through one projection: the smallest call a program makes,
        # all latency, launches and host work.
        {"name": "token", "kind": "apply", "m": 1, "k": HIDDEN, "n": HIDDEN, "bias": False, "columns": False,
         "graph": False},
        # The smallest prompt of the reference's own examples (128 tokens) through
        # one projection with a bias.
        {"name": "prompt_128", "kind": "apply", "m": 128, "k": HIDDEN, "n": HIDDEN, "bias": True, "columns": False,
         "graph": False},
        # A width that is a multiple of nothing, in the column layout that
        # linear_int8 returns: heads and adapters of other models.
        {"name": "odd_columns", "kind": "apply", "m": 333, "k": 1000, "n": 1111, "bias": True, "columns": True,
         "graph": False},
        # A 24-token question continued through a Gated DeltaNet layer and a GQA
        # layer, each with its FFN: the launch-bound inner loop, captured once
        # and replayed per question.
        {"name": "question_24", "kind": "layers", "m": 24, "layers": 2, "rank": 0, "graph": True},
        # The same question through a fine-tuned model: rank-16 adapters on every
        # projection.
        {"name": "question_24_lora", "kind": "layers", "m": 24, "layers": 2, "rank": 16, "graph": True},
        # 16 questions of 24 tokens stacked: a layer set's 9 projections in one
        # grouped call.
        {"name": "questions_384", "kind": "batch", "m": 384, "graph": False},
        # The FFN of a short prompt of ragged length, and of a 512-token prompt.
        {"name": "ffn_77", "kind": "ffn", "m": 77, "graph": False},
        {"name": "ffn_512", "kind": "ffn", "m": 512, "graph": False},
        # One layer of a 2048-token prefill (the headline workload is 24 of them).
        {"name": "prefill_2048", "kind": "layers", "m": 2048, "layers": 1, "rank": 0, "graph": False},
        # A 1000-token prompt through a layer with rank-16 adapters.
        {"name": "prefill_1000_lora", "kind": "layers", "m": 1000, "layers": 1, "rank": 16, "graph": False},
        # Two layers over the full 4096-token window, replayed.
        {"name": "prefill_4096", "kind": "layers", "m": 4096, "layers": 2, "rank": 0, "graph": True},
        # One stored BF16 weight made into a handle, and its first use: what a
        # program does for every projection when a model or an adapter set loads.
        {"name": "load_bf16", "kind": "load", "m": 24, "k": HIDDEN, "n": INTER, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("apply", "apply", "ffn", "layers", "layers", "batch", "load"))
    if kind == "apply":
        k, n = rng.choice(((HIDDEN, HIDDEN), (HIDDEN, KV), (HIDDEN, GDN_IN), (INTER, HIDDEN),
                           (_log_int(rng, 65, 6144), _log_int(rng, 17, 8224))))
        columns = rng.random() < 0.2
        return {"kind": kind, "m": _log_int(rng, 1, 4000), "k": k, "n": n, "bias": rng.random() < 0.5,
                "columns": columns, "graph": rng.random() < 0.3}
    if kind == "ffn":
        return {"kind": kind, "m": _log_int(rng, 1, 4000), "graph": rng.random() < 0.3}
    if kind == "layers":
        return {"kind": kind, "m": _log_int(rng, 4, 3000), "layers": rng.choice((1, 2)), "rank": rng.choice((0, 0, 16)),
                "graph": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": kind, "m": _log_int(rng, 8, 1024), "graph": rng.random() < 0.5}
    return {"kind": kind, "m": _log_int(rng, 1, 64), "k": _log_int(rng, 512, 6144), "n": _log_int(rng, 256, 8224),
            "dtype": rng.choice(("bf16", "f16", "f32"))}


# ---------------------------------------------------------------- inputs

_context = None


def _ctx():
    """The one context that a program keeps."""
    global _context
    if _context is None:
        _context = dq8.Context(0)
    return _context


class _Inputs:
    """Inputs made in one order from the seed alone."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")

    def acts(self, m, k):
        x = self.randn(m, k)
        hot = torch.randperm(k, generator=self.gen, device="cuda")[: max(1, k // 100)]
        x[:, hot] *= 20.0
        return x

    def weight(self, n, k):
        return self.randn(n, k) * 0.02

    def adapter(self, n, k, rank):
        return (self.randn(rank, k) * 0.02, self.randn(n, rank) * 0.05) if rank else None


def _layer_shapes(case, i):
    return GDN if i % 2 == 0 else GQA


def _tensors(case, seed):
    """A case's inputs as plain tensors: {"x": ..., "w": ...}, layers as lists of such."""
    g = _Inputs(seed)
    kind, m = case["kind"], case["m"]
    if kind == "apply":
        return {"x": g.acts(m, case["k"]), "w": g.weight(case["n"], case["k"]),
                "bias": g.randn(case["n"]) if case["bias"] else None}
    if kind == "load":
        dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[case["dtype"]]
        return {"x": g.acts(m, case["k"]), "w": g.weight(case["n"], case["k"]).to(dt)}
    if kind == "batch":
        shapes = GDN + GQA + (("o", HIDDEN, HIDDEN), ("out", HIDDEN, HIDDEN), ("gate", HIDDEN, INTER),
                              ("up", HIDDEN, INTER), ("down", INTER, HIDDEN))
        return {"shapes": shapes, "x": {k: g.acts(m, k) for k in (HIDDEN, INTER)},
                "w": [g.weight(n, k) for _, k, n in shapes]}
    rank = case.get("rank", 0)
    layers = []
    for i in range(case.get("layers", 1)):
        t = {"ffn_x": g.acts(m, HIDDEN), "residual": g.randn(m, HIDDEN), "w": {}, "ab": {}}
        shapes = (("gate", HIDDEN, INTER), ("up", HIDDEN, INTER), ("down", INTER, HIDDEN))
        if kind == "layers":
            t["x"], t["mixed"] = g.acts(m, HIDDEN), g.acts(m, HIDDEN)
            shapes = _layer_shapes(case, i) + (("out", HIDDEN, HIDDEN),) + shapes
        for name, k, n in shapes:
            t["w"][name], t["ab"][name] = g.weight(n, k), g.adapter(n, k, rank)
        layers.append(t)
    return {"layers": layers}


# ------------------------------------------------------------ preparation


def _quantized(ctx, m, k):
    return (torch.empty((m, k), dtype=torch.int8, device="cuda"),
            torch.empty((m, dq8.groups(k)), dtype=torch.float32, device="cuda"))


def _prepare_layer(ctx, case, t, flag):
    m, kind = case["m"], case["kind"]
    w = {name: ctx.weights_from_f32(v) for name, v in t["w"].items()}
    layer = {"w": w, "flag": flag, "ab": t["ab"], "ffn_x": t["ffn_x"], "residual": t["residual"],
             "h": torch.empty((m, INTER), device="cuda")}
    layer["q"] = _quantized(ctx, m, HIDDEN)
    if kind == "layers":
        layer["x"], layer["mixed"] = t["x"], t["mixed"]
        layer["first"] = [name for name in w if name not in ("out", "gate", "up", "down")]
        layer["outs"] = {name: torch.empty((m, w[name].n), device="cuda") for name in layer["first"] + ["out"]}
    layer["mids"] = {name: torch.empty((m, ab[0].shape[0]), device="cuda")
                     for name, ab in t["ab"].items() if ab is not None and name != "down"}
    return layer


def prepare(case, seed):
    ctx = _ctx()
    t = _tensors(case, seed)
    kind, m = case["kind"], case["m"]
    state = {"case": case, "ctx": ctx, "graph": None}
    if kind == "load":
        state["data"] = t["w"]
        state["q"] = ctx.quantize(t["x"])
        state["out"] = torch.empty((m, case["n"]), device="cuda")
        return state
    if kind == "apply":
        shape = (case["n"], m) if case["columns"] else (m, case["n"])
        state.update(x=t["x"], bias=t["bias"], w=ctx.weights_from_f32(t["w"]), out=torch.empty(shape, device="cuda"))
    elif kind == "batch":
        q = {k: ctx.quantize(x) for k, x in t["x"].items()}
        state["items"] = [
            dq8.Item(ctx.weights_from_f32(w), q[k][0], q[k][1], torch.empty((m, n), device="cuda"))
            for (_, k, n), w in zip(t["shapes"], t["w"])]
    else:
        flag = torch.zeros(1, dtype=torch.int32, device="cuda")
        state["layers"] = [_prepare_layer(ctx, case, lt, flag) for lt in t["layers"]]
    if case["graph"]:
        ctx.reserve(m, max(INTER, case.get("k", 0)), case.get("rank", 0))
        keep = [layer["residual"].clone() for layer in state.get("layers", ())]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(state)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            _pass(state)
        for layer, r in zip(state.get("layers", ()), keep):
            layer["residual"].copy_(r)
        state["graph"] = graph
    return state


# -------------------------------------------------------------- one pass


def _lora(layer, name):
    ab = layer["ab"][name]
    return None if ab is None else dq8.Lora(layer["mids"][name], ab[1], LORA_SCALE)


def _mids(ctx, layer, names, x):
    names = [n for n in names if layer["ab"][n] is not None]
    if names:
        ctx.lora_mid_batch([(x, layer["ab"][n][0]) for n in names], [layer["mids"][n] for n in names])


def _ffn(ctx, layer):
    w, (q, s), x = layer["w"], layer["q"], layer["ffn_x"]
    ctx.quantize(x, q, s, nonfinite=layer["flag"])
    _mids(ctx, layer, ("gate", "up"), x)
    down = layer["ab"]["down"]
    ctx.ffn(w["gate"], w["up"], w["down"], q, s, layer["residual"], h=layer["h"], gate_lora=_lora(layer, "gate"),
            up_lora=_lora(layer, "up"), down_lora=None if down is None else (down[0], down[1], LORA_SCALE))


def _layer(ctx, layer):
    w, (q, s) = layer["w"], layer["q"]
    for names, x in ((layer["first"], layer["x"]), (["out"], layer["mixed"])):
        ctx.quantize(x, q, s, nonfinite=layer["flag"])
        _mids(ctx, layer, names, x)
        ctx.linear_batch([dq8.Item(w[n], q, s, layer["outs"][n], lora=_lora(layer, n)) for n in names])
    _ffn(ctx, layer)


def _pass(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "apply":
        ctx.apply(state["w"], state["x"], out=state["out"], bias=state["bias"],
                  layout=dq8.COLUMNS if case["columns"] else dq8.ROWS)
    elif kind == "batch":
        ctx.linear_batch(state["items"])
    elif kind == "ffn":
        _ffn(ctx, state["layers"][0])
    else:
        for layer in state["layers"]:
            _layer(ctx, layer)


def run(state):
    if state["case"]["kind"] == "load":
        state["w"] = state["ctx"].weights_from_raw(state["data"])
        return state["ctx"].linear(state["w"], *state["q"], out=state["out"])
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        _pass(state)
    if "items" in state:
        return [it.out for it in state["items"]]
    if "layers" in state:
        return [dict(layer.get("outs", {}), h=layer["h"], residual=layer["residual"]) for layer in state["layers"]]
    return state["out"]


# ------------------------------------------------------------------ work


def _linear_work(m, k, n, rank=0):
    g = dq8.groups(k)
    return {"flops": 2.0 * m * k * n + 2.0 * m * rank * (k + n),
            "bytes": n * k + 4.0 * n * g + 4.0 * m * n + 4.0 * rank * (k + n)}


def work(case):
    kind, m = case["kind"], case["m"]
    parts, act = [], 0.0
    if kind in ("apply", "load"):
        parts = [_linear_work(m, case["k"], case["n"])]
        act = 4.0 * m * case["k"]
        if kind == "load":  # the stored elements in; the handle written and read once
            size = 4 if case["dtype"] == "f32" else 2
            act = m * case["k"] * 1.0625 + case["n"] * case["k"] * (size + 1.0625)
    elif kind == "batch":
        shapes = GDN + GQA + (("", HIDDEN, HIDDEN),) * 2 + (("", HIDDEN, INTER),) * 2 + (("", INTER, HIDDEN),)
        parts = [_linear_work(m, k, n) for _, k, n in shapes]
        act = 1.0625 * m * (HIDDEN + INTER)
    else:
        rank = case.get("rank", 0)
        for i in range(case.get("layers", 1)):
            shapes = (("", HIDDEN, INTER), ("", INTER, HIDDEN))
            act += 4.0 * m * (HIDDEN + HIDDEN)  # the FFN's input, the old residual
            if kind == "layers":
                shapes = _layer_shapes(case, i) + (("", HIDDEN, HIDDEN),) + shapes
                act += 4.0 * m * (HIDDEN + HIDDEN)
            parts += [_linear_work(m, k, n, rank) for _, k, n in shapes]
            gate = _linear_work(m, HIDDEN, INTER, rank)  # h is written once for gate and up
            gate["bytes"] -= 4.0 * m * INTER
            parts.append(gate)
    return {"bytes": act + sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def tolerance(case):
    return "exact"


# --------------------------------------------------------- 64-bit results


def _format(x):
    """The int8 format of fp32 values [r][k], as its definition has it (absmax / 127 per group of 64, at
    least the smallest normal, 1 for zeros; the nearest integer, halves away from zero), back in 64 bits."""
    r, k = x.shape
    pad = (-k) % 64
    v = torch.nn.functional.pad(x, (0, pad)).reshape(r, -1, 64)
    top = v.abs().amax(2, keepdim=True)
    # (by a tensor: torch divides by a number through its reciprocal, which is not the rounded quotient)
    scale = (top / torch.full_like(top, 127.0)).clamp_min(torch.finfo(torch.float32).tiny)
    scale = torch.where(top == 0, torch.ones_like(top), scale)
    ratio = (v / scale).double()
    q = (torch.sign(ratio) * torch.floor(ratio.abs() + 0.5)).clamp(-127, 127)
    return (q * scale.double()).reshape(r, -1)[:, :k].contiguous()


def _linear64(xq, w, ab=None, x=None):
    y = xq @ _format(w).t().contiguous()
    if ab is not None:
        mid = x.double() @ ab[0].double().t().contiguous()
        y = y + LORA_SCALE * (mid @ ab[1].double().t().contiguous())
    return y


def exact(case, seed):
    t = _tensors(case, seed)
    kind = case["kind"]
    if kind in ("apply", "load"):
        y = _linear64(_format(t["x"]), t["w"].float())
        if t.get("bias") is not None:
            y = y + t["bias"].double()
        return y.t().contiguous() if case.get("columns") else y
    if kind == "batch":
        xq = {k: _format(x) for k, x in t["x"].items()}
        return [_linear64(xq[k], w) for (_, k, _), w in zip(t["shapes"], t["w"])]
    out = []
    for i, lt in enumerate(t["layers"]):
        w, ab, got = lt["w"], lt["ab"], {}
        if kind == "layers":
            xq, mq = _format(lt["x"]), _format(lt["mixed"])
            for name, _, _ in _layer_shapes(case, i):
                got[name] = _linear64(xq, w[name], ab[name], lt["x"])
            got["out"] = _linear64(mq, w["out"], ab["out"], lt["mixed"])
        fq = _format(lt["ffn_x"])
        gate, up = (_linear64(fq, w[n], ab[n], lt["ffn_x"]) for n in ("gate", "up"))
        got["h"] = gate * torch.sigmoid(gate) * up
        h = got["h"].float()
        got["residual"] = lt["residual"].double() + _linear64(_format(h), w["down"], ab["down"], h)
        out.append(got)
    return out
