"""The work a user of the MoE layer has it do, as cases that can be timed and compared.

Kinds of call, each through a public entry point of ``veymoe``:

* ``step``     one decode step through a stack of layers, replayed as one graph (``StepGraph``): 1 to 8 tokens;
* ``layer``    ``MoELayer`` calls, one per layer of a short stack: single tokens, batched decode, prefill chunks and
               layer-major windows;
* ``experts``  the expert block alone (``HipSwitchGLU``) on given routes, one output row per token and slot;
* ``hyper``    the hyper-connection in front of a decoder's MoE branch (``HyperConnection``).

Layer widths: the small layer (hidden 1024, intermediate 256, 64 experts top-4, no shared expert), the full-size layer
(2048 / 512, 512 experts top-10 and a shared expert) and the checkpoint's widths (2560 / 640, the same routing).
Weights are uniform nibbles with scales U(0.005, 0.02) and biases U(-0.1, 0.1) in bf16, activations N(0, 1) bf16;
a skewed router adds log Zipf(1.1) popularity to its logits, as decode batches meet it.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "veystrix-core_amd"))

# name: hidden, intermediate, experts, top_k, shared expert
WIDTHS = {"small": (1024, 256, 64, 4, False), "full": (2048, 512, 512, 10, True), "wide": (2560, 640, 512, 10, True)}
EPS = 1e-6
STREAMS, LOWRANK = 4, 32


def listed():
    return [
        # one token through one small layer, called eagerly: the smallest call, latency and launches
        {"name": "token_small", "kind": "layer", "width": "small", "rows": 1, "layers": 1, "zipf": False},
        # decode at batch 1, the step of a serving loop
        {"name": "step_full_1", "kind": "step", "width": "full", "rows": 1, "layers": 12, "zipf": False},
        {"name": "step_wide_1", "kind": "step", "width": "wide", "rows": 1, "layers": 8, "zipf": False},
        # a handful of tokens at once: speculative verification or a few requests
        {"name": "step_wide_5", "kind": "step", "width": "wide", "rows": 5, "layers": 4, "zipf": False},
        # batched decode with skewed expert popularity
        {"name": "batch_full_32", "kind": "layer", "width": "full", "rows": 32, "layers": 4, "zipf": True},
        {"name": "batch_wide_24", "kind": "layer", "width": "wide", "rows": 24, "layers": 4, "zipf": True},
        # a short prompt, ragged
        {"name": "prompt_wide_333", "kind": "layer", "width": "wide", "rows": 333, "layers": 1, "zipf": False},
        # prefill chunks
        {"name": "prefill_full_2048", "kind": "layer", "width": "full", "rows": 2048, "layers": 1, "zipf": False},
        {"name": "prefill_wide_1999", "kind": "layer", "width": "wide", "rows": 1999, "layers": 1, "zipf": False},
        # a layer-major window of four chunks
        {"name": "window_full_8192", "kind": "layer", "width": "full", "rows": 8192, "layers": 1, "zipf": False},
        # the expert block alone, a caller that routes by itself
        {"name": "experts_small_700", "kind": "experts", "width": "small", "rows": 700, "layers": 1, "zipf": False},
        # the decoder glue in front of a prefill chunk's MoE call
        {"name": "hyper_wide_700", "kind": "hyper", "width": "wide", "rows": 700, "layers": 1, "zipf": False},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(("layer", "step", "experts", "hyper"), (6, 2, 1, 1))[0]
    width = rng.choice(("small", "full", "full", "wide", "wide"))
    layers, zipf = 1, False
    if kind == "step":
        rows, layers = _log(rng, 1, 8), rng.randint(3, 8)
        zipf = rng.random() < 0.3
    elif kind == "layer":
        rows = _log(rng, 1, 4096 if width == "wide" else 8192)
        layers = rng.randint(1, 3) if rows <= 64 else 1
        zipf = rng.random() < (0.7 if rows <= 256 else 0.2)
    elif kind == "experts":
        rows = _log(rng, 1, 2048)
        zipf = rng.random() < 0.3
    else:
        rows = _log(rng, 1, 4096)
    return {"kind": kind, "width": width, "rows": rows, "layers": layers, "zipf": zipf}


# ------------------------------------------------------------------ inputs --

def _q4(shape, gen):
    """(words, scales, biases) of a Q4/G32 projection [.., out, in]."""
    lead, width = tuple(shape[:-1]), shape[-1]
    w = torch.randint(-2 ** 31, 2 ** 31, (*lead, width // 8), dtype=torch.int32, device="cuda", generator=gen)
    s = torch.empty((*lead, width // 32), device="cuda").uniform_(0.005, 0.02, generator=gen).bfloat16()
    b = torch.empty((*lead, width // 32), device="cuda").uniform_(-0.1, 0.1, generator=gen).bfloat16()
    return w, s, b


def _parts(hidden, inter):
    """(first byte, bytes, out width, in width, is words) of a record's nine parts: gate, up, down by words, scales, biases."""
    at, parts = 0, []
    for out_w, in_w in ((inter, hidden), (inter, hidden), (hidden, inter)):
        for words in (True, False, False):
            size = out_w * in_w // 2 if words else out_w * in_w // 32 * 2
            parts.append((at, size, out_w, in_w, words))
            at += size
    return parts, at


def _fill_records(records, hidden, inter, gen):
    """Random experts in a [n, stride] byte view of whole records."""
    n = records.shape[0]
    parts, _ = _parts(hidden, inter)
    records.view(torch.int32).random_(-2 ** 31, 2 ** 31, generator=gen)
    for i, (at, size, _, _, words) in enumerate(parts):
        if not words:
            low, high = (0.005, 0.02) if i % 3 == 1 else (-0.1, 0.1)
            v = torch.empty((n, size // 2), device="cuda").uniform_(low, high, generator=gen)
            records[:, at:at + size].view(torch.bfloat16).copy_(v)


def _router(case, layer, seed, gen):
    hidden, _, experts, _, _ = WIDTHS[case["width"]]
    weight = (torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02).bfloat16()
    bias = None
    if case["zipf"]:
        pmf = np.arange(1, experts + 1, dtype=np.float64) ** -1.1
        perm = np.random.default_rng([seed & 0xFFFFFFFF, layer]).permutation(experts)
        bias = np.empty(experts, dtype=np.float32)
        bias[perm] = np.log(pmf / pmf.sum())
        bias = torch.from_numpy(bias).cuda()
    return weight, bias


def _activations(rows, width, gen):
    return torch.randn((rows, width), device="cuda", generator=gen).bfloat16()


def _layer_inputs(case, seed, records):
    """The stack's inputs; the experts go into ``records`` [layers * experts, stride] in a random slot order."""
    hidden, inter, experts, _, shared = WIDTHS[case["width"]]
    layers = case["layers"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    for at in range(0, records.shape[0], experts):
        _fill_records(records[at:at + experts], hidden, inter, gen)
    slots = np.random.default_rng([seed & 0xFFFFFFFF, 7]).permutation(layers * experts).astype(np.int32)
    got = []
    for layer in range(layers):
        router, bias = _router(case, layer, seed, gen)
        one = {"router": router, "bias": bias, "slots": slots[layer * experts:(layer + 1) * experts],
               "x": _activations(case["rows"], hidden, gen)}
        if shared:
            one["shared"] = [_q4((1, inter, hidden), gen), _q4((1, inter, hidden), gen), _q4((1, hidden, inter), gen)]
            one["shared_gate"] = _q4((1, 1, hidden), gen)
        got.append(one)
    return got


def _experts_inputs(case, seed):
    """Dense experts, activations and the routes of a caller's own router."""
    hidden, inter, experts, top_k, _ = WIDTHS[case["width"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    proj = [_q4((experts, inter, hidden), gen), _q4((experts, inter, hidden), gen), _q4((experts, hidden, inter), gen)]
    router, bias = _router(case, 0, seed, gen)
    x = _activations(case["rows"], hidden, gen)
    logits = x.float() @ router.float().t()
    inds = (logits if bias is None else logits + bias).topk(top_k, dim=-1).indices.to(torch.int32)
    return proj, x, inds


def _hyper_inputs(case, seed):
    hidden = WIDTHS[case["width"]][0]
    n = STREAMS * hidden
    gen = torch.Generator(device="cuda").manual_seed(seed)
    gain = (1.0 + 0.1 * torch.randn((n,), device="cuda", generator=gen)).bfloat16()

    def proj(out_w, in_w):  # outputs of order one, with zero-mean weights
        w = torch.randint(-2 ** 31, 2 ** 31, (out_w, in_w // 8), dtype=torch.int32, device="cuda", generator=gen)
        s = torch.empty((out_w, in_w // 32), device="cuda").uniform_(0.5, 1.0, generator=gen) / (4 * math.sqrt(in_w))
        return w, s.bfloat16(), (-7.5 * s).bfloat16()

    down, up, inject = proj(LOWRANK, n), proj(n, LOWRANK), proj(STREAMS, n)
    return gain, down, up, inject, _activations(case["rows"], n, gen)


# ------------------------------------------------------------------- calls --

def _projection(q4):
    from veymoe.executor import Q4G32Projection

    return Q4G32Projection(*q4)


def prepare(case, seed):
    from veymoe.layer import HipSwitchGLU, MoELayer, QuantizedMLP, RouterLinear
    from veymoe.layout import RecordLayout
    from veymoe.pool import ExpertPool

    hidden, inter, experts, top_k, _ = WIDTHS[case["width"]]
    if case["kind"] == "hyper":
        from veymoe.glue import HyperConnection

        gain, down, up, inject, x = _hyper_inputs(case, seed)
        return {"kind": "hyper", "x": x,
                "hyper": HyperConnection(gain, _projection(down), _projection(up), _projection(inject), STREAMS,
                                         eps=EPS)}
    if case["kind"] == "experts":
        proj, x, inds = _experts_inputs(case, seed)
        names = ("gate_proj", "up_proj", "down_proj")
        block = HipSwitchGLU(hidden, inter, experts, layer_id=1,
                             projections={n: _projection(p) for n, p in zip(names, proj)})
        return {"kind": "experts", "x": x, "inds": inds, "block": block}
    layout = RecordLayout(hidden, inter)
    layers = case["layers"]
    pool = ExpertPool(layout, layers * experts, layers=layers, experts=experts)
    inputs = _layer_inputs(case, seed, pool.buffer[pool.header_size:].view(layers * experts, layout.record_stride))
    stack = []
    for i, one in enumerate(inputs):
        pool.place_all(i, one["slots"])
        shared = gate = None
        if "shared" in one:
            shared = QuantizedMLP(*[_projection(p) for p in one["shared"]])
            gate = _projection(one["shared_gate"])
        block = HipSwitchGLU(hidden, inter, experts, pool=pool, layer_id=i)
        stack.append(MoELayer(RouterLinear(one["router"], one["bias"]), block, top_k, shared_expert=shared,
                              shared_expert_gate=gate))
    pool.sync_tables()
    if case["kind"] == "step":
        from veymoe.graph import StepGraph

        return {"kind": "step", "x": torch.stack([one["x"] for one in inputs]),
                "step": StepGraph(stack, rows=case["rows"]).capture()}
    return {"kind": "layer", "x": [one["x"] for one in inputs], "stack": stack}


def run(state):
    kind = state["kind"]
    if kind == "step":
        return state["step"].replay(state["x"])
    if kind == "layer":
        return [layer(x) for layer, x in zip(state["stack"], state["x"])]
    if kind == "experts":
        return state["block"](state["x"], state["inds"])
    mixed, _, weights = state["hyper"](state["x"])
    return mixed, weights


# -------------------------------------------------------------------- work --

def _distinct(case):
    """Distinct experts that a call's rows route to, from random logits of the case's distribution."""
    hidden, _, experts, top_k, _ = WIDTHS[case["width"]]
    rng = np.random.default_rng(1)
    logits = rng.normal(0.0, 0.02 * math.sqrt(hidden), (min(case["rows"], 1024), experts))
    if case["zipf"]:
        logits = logits - 1.1 * np.log(np.arange(1, experts + 1))
    return len(np.unique(np.argpartition(-logits, top_k - 1, axis=1)[:, :top_k]))


def work(case):
    hidden, inter, experts, top_k, shared = WIDTHS[case["width"]]
    rows = case["rows"]
    if case["kind"] == "hyper":
        n = STREAMS * hidden
        weights = n * (LOWRANK * 2 + STREAMS) * 5 // 8 + 2 * n
        return {"bytes": weights + 2 * rows * (n + hidden + STREAMS), "flops": 2 * rows * n * (2 * LOWRANK + STREAMS)}
    expert = 15 * hidden * inter // 8
    outs = top_k if case["kind"] == "experts" else 1
    moved = _distinct(case) * expert + 2 * rows * hidden * (1 + outs)
    flops = 6 * rows * top_k * hidden * inter
    if case["kind"] == "experts":
        moved += 4 * rows * top_k
    else:
        moved += 2 * experts * hidden
        flops += 2 * rows * experts * hidden
        if shared:
            moved += expert + hidden * 5 // 8
            flops += rows * (6 * hidden * inter + 2 * hidden)
    return {"bytes": case["layers"] * moved, "flops": case["layers"] * flops}


def tolerance(case):
    # bf16 outputs, and bf16 rounding at every step inside: against 64 bits the outputs are 2e-3 to 5e-3 off
    return {"rel": 1e-2, "max": 0.2}


# ------------------------------------------------------------------- exact --

def _dense(w, s, b):
    """Q4/G32 words, scales and biases as 64-bit weights [.., out, in]."""
    shifts = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> shifts) & 15).double().reshape(*s.shape, 32)
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(*s.shape[:-1], -1)


def _swiglu(x, gate, up, down):
    return (torch.nn.functional.silu(x @ _dense(*gate).t()) * (x @ _dense(*up).t())) @ _dense(*down).t()


def _record(record, hidden, inter):
    parts, _ = _parts(hidden, inter)
    got = [record[at:at + size].view(torch.int32 if words else torch.bfloat16).view(out_w, -1)
           for at, size, out_w, _, words in parts]
    return got[:3], got[3:6], got[6:]


def _routes(x, router, bias, top_k):
    """The layer's selection: bf16 logits and gates, the larger gate first and the lower expert on ties."""
    logits = x.double() @ router.double().t()
    if bias is not None:
        logits = logits + bias.double()
    gates = torch.softmax(logits.bfloat16().double(), dim=-1)
    order = torch.sort(gates.bfloat16().float(), dim=-1, descending=True, stable=True).indices[:, :top_k]
    scores = torch.gather(gates, 1, order)
    return order, scores / scores.sum(-1, keepdim=True)


def exact(case, seed):
    hidden, inter, experts, top_k, _ = WIDTHS[case["width"]]
    rows = case["rows"]
    if case["kind"] == "hyper":
        gain, down, up, inject, x = _hyper_inputs(case, seed)
        x = x.double()
        normed = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain.double()
        mix = torch.sigmoid(torch.nn.functional.silu(normed @ _dense(*down).t() / STREAMS) @ _dense(*up).t())
        mixed = (mix * normed).reshape(rows, STREAMS, hidden).mean(1)
        return mixed, 2 * torch.sigmoid(normed @ _dense(*inject).t() / STREAMS)
    if case["kind"] == "experts":
        proj, x, inds = _experts_inputs(case, seed)
        out = torch.zeros((rows, top_k, hidden), dtype=torch.float64, device="cuda")
        for e in torch.unique(inds).tolist():
            row, slot = torch.nonzero(inds == e, as_tuple=True)
            out[row, slot] = _swiglu(x[row].double(), *[[part[e] for part in p] for p in proj])
        return out
    _, stride = _parts(hidden, inter)
    records = torch.empty((case["layers"] * experts, stride), dtype=torch.uint8, device="cuda")
    outs = []
    for one in _layer_inputs(case, seed, records):
        x = one["x"].double()
        inds, scores = _routes(one["x"], one["router"], one["bias"], top_k)
        out = torch.zeros((rows, hidden), dtype=torch.float64, device="cuda")
        for e in torch.unique(inds).tolist():
            row, slot = torch.nonzero(inds == e, as_tuple=True)
            y = _swiglu(x[row], *_record(records[int(one["slots"][e])], hidden, inter))
            out[row] += scores[row, slot].unsqueeze(-1) * y
        if "shared" in one:
            gate = torch.sigmoid(x @ _dense(*one["shared_gate"])[0].t())
            out += gate * _swiglu(x, *[[part[0] for part in p] for p in one["shared"]])
        outs.append(out)
    return torch.stack(outs) if case["kind"] == "step" else outs
