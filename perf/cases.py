"""The work that programs on this package have it do, as cases that can be timed and compared.

A case is a dict of plain values. `listed` names the ones that stand for the package's use, `draw` gives more of
the same ranges, `prepare` makes what a program holds before the call (weights on the device, inputs, layers and,
for decode, the captured graph of a token's pass), `run` is one pass through the public entry points, `exact` the
same outputs in 64 bits, and `work` and `tolerance` say what a pass cannot do without and how far two correct
results may lie apart.

Four kinds of pass:
- dense: `QMatMul.forward` over `calls` different matrices (a model's projections, one after another);
- moe: `MoeLayer.forward` over a chain of `layers` layers, every expert resident, or `slots` of them behind a slot
  table. Decode steps (graph = True) run as serving programs run them, one captured graph per step;
- block: a whole MoE block eagerly: router logits, routed experts, and the shared expert added to them;
- shrink: the re-encoding of a layer's experts to Q2_K.
"""
import base64
import math

import numpy as np
import torch

from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth

# ------------------------------------------------------------------------------ the cases


def _moe(name, gate_up, down, experts, top_k, hidden, inter, tokens, layers, slots=0, act="silu", rows16=False):
    return {"name": name, "kind": "moe", "gate_up": gate_up, "down": down, "experts": experts, "slots": slots, "top_k": top_k,
            "hidden": hidden, "inter": inter, "act": act, "rows16": rows16, "tokens": tokens, "layers": layers, "graph": tokens <= 8}


def _dense(name, weight, n, k, rows, calls):
    return {"name": name, "kind": "dense", "weight": weight, "n": n, "k": k, "rows": rows, "calls": calls, "graph": rows <= 16}


def listed():
    return [
        # the smallest calls: one token through 32 small projections
        _dense("dense_q8_0_1row", "q8_0", 2048, 2048, 1, 32),
        # 16 sequences decoded together through an attention-sized projection
        _dense("dense_q4k_16rows", "q4_K", 4096, 4096, 16, 16),
        # a prompt's chunk of 512 tokens through the same projection
        _dense("dense_q4k_512rows", "q4_K", 4096, 4096, 512, 8),
        # a short prompt through one of the matrices that 4-bit mixes keep in Q6_K: ragged rows of x and of W
        _dense("dense_q6k_77rows", "q6_K", 4001, 4096, 77, 4),
        # one token through half of a 40-layer model of 256 small 2-bit experts, top-8
        _moe("moe_iq2_decode", "iq2_xxs", "iq2_s", 256, 8, 2048, 512, 1, 20),
        # one token through the experts of a 12-layer MXFP4 model, laid out in row groups when loaded
        _moe("moe_mxfp4_decode", "mxfp4", "mxfp4", 128, 4, 2880, 2880, 1, 12, act="clamped", rows16=True),
        # one token through layers that hold 56 of their 512 experts in a bank
        _moe("moe_bank_decode", "iq3_s", "q4_K", 512, 10, 2048, 512, 1, 20, slots=56),
        # 8 sequences decoded together
        _moe("moe_iq2_8tokens", "iq2_xxs", "iq2_s", 256, 8, 2048, 512, 8, 8),
        # a prompt of 1,500 tokens through a layer of small 2-bit experts
        _moe("moe_iq2_prefill", "iq2_xxs", "iq2_s", 256, 8, 2048, 512, 1500, 1),
        # a prompt of 2,048 tokens through an MXFP4 layer: the largest pass
        _moe("moe_mxfp4_prefill", "mxfp4", "mxfp4", 128, 4, 2880, 2880, 2048, 1, act="clamped", rows16=True),
        # a short prompt (odd length) through a whole block of a 4-bit mix: Q4_K gate and up, Q6_K down, Q8_0 shared expert
        dict(_moe("block_kquant_301tokens", "q4_K", "q6_K", 128, 8, 2048, 768, 301, 1), kind="block", shared="q8_0", shared_inter=512),
        # 32 experts re-encoded on arrival: gate and up from Q3_K, down from Q5_K
        {"name": "shrink_32experts", "kind": "shrink", "experts": 32, "hidden": 2048, "inter": 512, "weighted": False},
    ]


# expert formats that are used together: (gate and up, down)
_PAIRS = [("iq2_xxs", "iq2_s"), ("iq2_xxs", "iq3_s"), ("iq2_s", "iq3_s"), ("iq3_s", "q4_K"), ("iq3_xxs", "iq4_xs"), ("iq4_xs", "iq4_xs"),
          ("q2_K", "q2_K"), ("q4_K", "q4_K"), ("q4_K", "q6_K"), ("q5_K", "q6_K"), ("q8_0", "q8_0"), ("mxfp4", "mxfp4")]
_DENSE = ["q8_0", "q8_0", "q2_K", "q4_K", "q4_K", "q4_K", "q5_K", "q6_K", "q6_K", "iq2_xxs", "iq2_s", "iq3_xxs", "iq3_s", "iq4_xs", "mxfp4"]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.random()
    if what < 0.35:
        weight = rng.choice(_DENSE)
        k = 32 * _log_int(rng, 16, 256) if weight in ("q8_0", "mxfp4") else 256 * _log_int(rng, 2, 32)
        n, rows = _log_int(rng, 256, 8192), _log_int(rng, 1, 1024)
        calls = max(1, min(16, int(2e8 / (F.matrix_bytes(F.BY_NAME[weight], n, k) + 4 * rows * (n + k)))))
        return {k_: v for k_, v in _dense("", weight, n, k, rows, calls).items() if k_ != "name"}
    if what < 0.92:
        gate_up, down = rng.choice(_PAIRS)
        mx = gate_up == "mxfp4"
        hidden = 32 * rng.randint(32, 96) if mx else 256 * rng.randint(4, 12)
        inter = 32 * rng.randint(16, 90) if mx else 256 * rng.randint(1, 6)
        top_k = rng.randint(2, 10)
        tokens = _log_int(rng, 1, 1024)
        one = _expert_bytes(gate_up, down, hidden, inter)
        experts = max(4 * top_k, min(_log_int(rng, 32, 512), int(1.5e9 / one)))
        slots = max(top_k, experts // rng.randint(2, 8)) if rng.random() < 0.2 else 0
        layers = max(1, min(8, int(4e9 / ((slots or experts) * one)))) if tokens <= 8 else 1
        c = _moe("", gate_up, down, experts, top_k, hidden, inter, tokens, layers, slots, "clamped" if mx else "silu", mx and rng.random() < 0.6)
        if not mx and not slots and tokens > 8 and rng.random() < 0.3:
            c.update(kind="block", shared=rng.choice(["q8_0", "q4_K", "q6_K"]), shared_inter=256 * rng.randint(1, 4))
        del c["name"]
        return c
    return {"kind": "shrink", "experts": _log_int(rng, 1, 64), "hidden": 256 * rng.randint(4, 12), "inter": 256 * rng.randint(1, 6),
            "weighted": rng.random() < 0.5}


def _expert_bytes(gate_up, down, hidden, inter):
    g, d = F.BY_NAME[gate_up], F.BY_NAME[down]
    return 2 * F.matrix_bytes(g, inter, hidden) + F.matrix_bytes(d, hidden, inter)


# ------------------------------------------------------------------------------ inputs (of the seed alone)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


def _blocks(dtype, weights, gen):
    return synth.device_blocks(dtype, weights, gen, "cuda")


def _dense_inputs(c, gen):
    x = _randn(gen, c["calls"], c["rows"], c["k"])
    dt = F.BY_NAME[c["weight"]]
    for i in range(c["calls"]):
        yield _blocks(dt, c["n"] * c["k"], gen), x[i]


def _moe_inputs(c, gen):
    """Per layer: the three banks' GGUF blocks, the biases, the experts held in the slots, x and the router logits (or the
    router's and the shared expert's weights)."""
    h, i, e, t = c["hidden"], c["inter"], c["experts"], c["tokens"]
    held = c["slots"] or e
    dts = [F.BY_NAME[c["gate_up"]]] * 2 + [F.BY_NAME[c["down"]]]
    shapes = [(i, h), (i, h), (h, i)]
    for _ in range(c["layers"]):
        d = {"raw": [_blocks(dts[m], held * shapes[m][0] * shapes[m][1], gen) for m in range(3)], "dtypes": dts, "shapes": shapes}
        d["bias"] = [0.02 * _randn(gen, e, i), 0.02 * _randn(gen, e, i), 0.02 * _randn(gen, e, h)] if c["act"] == "clamped" else None
        d["x"] = _randn(gen, t, h)
        if c["act"] == "clamped":
            d["x"] = d["x"].to(torch.bfloat16).float()
        d["resident"] = None
        if c["kind"] == "block":
            # router rows of norm 1: logits of about N(0, 1)
            d["router"] = _randn(gen, e, h) / math.sqrt(h)
            s, si = F.BY_NAME[c["shared"]], c["shared_inter"]
            d["shared"] = [(_blocks(s, n * k, gen), s, (n, k)) for n, k in ((si, h), (si, h), (h, si))]
            d["gate_inp"] = _randn(gen, h) / math.sqrt(h)
        else:
            d["logits"] = _randn(gen, t, e)
            if c["slots"]:
                # the routing is restricted to the experts that the bank holds
                d["resident"] = torch.randperm(e, generator=gen, device="cuda")[:held]
                mask = torch.full((e,), -1e30, device="cuda")
                mask[d["resident"]] = 0.0
                d["logits"] = d["logits"] + mask
        yield d


def _shrink_inputs(c, gen):
    h, i, e = c["hidden"], c["inter"], c["experts"]
    for src, n, k in ((F.Q3_K, i, h), (F.Q3_K, i, h), (F.Q5_K, h, i)):
        yield src, _blocks(src, e * n * k, gen), e * n * k // 256, (_randn(gen, k).square() if c["weighted"] else None), k // 256


# ------------------------------------------------------------------------------ a program's state and its pass


def _moe_layer(c, d):
    banks = []
    for raw, dt, (n, k) in zip(d["raw"], d["dtypes"], d["shapes"]):
        b = ops.ExpertBank(raw, dt, n, k, c["slots"] or c["experts"], F.matrix_bytes(dt, n, k))
        banks.append(b.rows16() if c["rows16"] else b)
    table = None
    if d["resident"] is not None:
        table = torch.full((c["experts"],), -1, dtype=torch.int32, device="cuda")  # the bits of NO_SLOT
        table[d["resident"]] = torch.arange(c["slots"], dtype=torch.int32, device="cuda")
    act = ops.ExpertAct.clamped_swiglu(1.702, 7.0, *d["bias"]) if c["act"] == "clamped" else ops.ExpertAct.silu()
    return ops.MoeLayer(*banks, n_experts=c["experts"], top_k=c["top_k"], norm_topk_prob=True, act=act, slot_table=table)


def _pass(s):
    c = s["case"]
    if c["kind"] == "dense":
        return [m.forward(x) for m, x in s["calls"]]
    if c["kind"] == "moe":
        return [layer.forward(x, logits) for layer, x, logits in s["layers"]]
    if c["kind"] == "block":
        got = []
        for layer, shared, router, x in s["layers"]:
            logits = ops.router_logits(router, x)
            out, ids, w = layer.forward(x, logits)
            got.append((shared.forward(x, out), ids, w, logits))
        return got
    return [ops.requant_q2k(src, raw, blocks, shape, per_row) for src, raw, blocks, shape, per_row in s["matrices"]]


def prepare(case, seed):
    gen, s = _gen(seed), {"case": case, "graph": None}
    if case["kind"] == "dense":
        dt, shape = F.BY_NAME[case["weight"]], (case["n"], case["k"])
        s["calls"] = [(ops.QMatMul(ops.QTensor(raw, dt, shape)), x) for raw, x in _dense_inputs(case, gen)]
    elif case["kind"] == "shrink":
        s["matrices"] = list(_shrink_inputs(case, gen))
    else:
        s["layers"] = []
        for d in _moe_inputs(case, gen):
            layer = _moe_layer(case, d)
            if case["kind"] == "block":
                shared = ops.SharedExpert(*[ops.QTensor(*q) for q in d["shared"]], gate_inp=d["gate_inp"])
                s["layers"].append((layer, shared, d["router"], d["x"]))
            else:
                s["layers"].append((layer, d["x"], d["logits"]))
    if case.get("graph"):
        _pass(s)  # the layers' workspaces are made by their first call
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = _pass(s)
    return s


def run(state):
    if state["graph"] is None:
        return _pass(state)
    state["graph"].replay()
    return state["out"]


# ------------------------------------------------------------------------------ what a pass cannot do without


def work(case):
    c = case
    if c["kind"] == "dense":
        w = F.matrix_bytes(F.BY_NAME[c["weight"]], c["n"], c["k"])
        return {"bytes": c["calls"] * (w + 4 * c["rows"] * (c["n"] + c["k"])), "flops": 2 * c["calls"] * c["rows"] * c["n"] * c["k"]}
    if c["kind"] == "shrink":
        weights = c["experts"] * c["hidden"] * c["inter"] // 256
        # a minimum and a maximum, and two weighted fits of 16 values each: about 40 operations per weight
        return {"bytes": weights * (2 * 110 + 176 + 3 * 84), "flops": 3 * 256 * 40 * weights}
    t, e, h = c["tokens"], c["experts"], c["hidden"]
    held = c["slots"] or e
    picked = held * (1 - (1 - c["top_k"] / held) ** t)  # experts that some token picks, on average
    b = picked * _expert_bytes(c["gate_up"], c["down"], h, c["inter"]) + 4 * t * (2 * h + e) + 8 * t * c["top_k"]
    f = 6 * t * c["top_k"] * h * c["inter"]
    if c["kind"] == "block":
        b += 4 * e * h + _expert_bytes(c["shared"], c["shared"], h, c["shared_inter"]) + 4 * h
        f += 2 * t * e * h + 6 * t * h * c["shared_inter"]
    return {"bytes": c["layers"] * b, "flops": c["layers"] * f}


# What the entry points state: f32 activations in the matvecs (from 1 row, to 7 or, for Q4_K, 1) and for the formats without
# a matrix-core kernel; fp16 activations (2^-11 per value) in the others; three FP6 terms for MXFP4 experts.
_F32, _F16, _FP6X3 = {"rel": 2e-6}, {"rel": 1.5e-3}, {"rel": 1e-4}


def _dense_f16(dtype, rows):
    return dtype not in ("q5_K", "q6_K") and rows >= (2 if dtype == "q4_K" else 8)


def tolerance(case):
    c = case
    if c["kind"] == "shrink":
        return "exact"
    if c["kind"] == "dense":
        return dict(_F16 if _dense_f16(c["weight"], c["rows"]) else _F32)
    grouped = c["tokens"] >= 16 and not {c["gate_up"], c["down"]} & {"q5_K", "q6_K"}
    t = _F32 if not grouped else _FP6X3 if c["gate_up"] == "mxfp4" else _F16
    if c["kind"] == "block" and t is _F32:
        # the router's f32 logits are 1e-6 off, and so the weights. The shared expert's fp16 shows beside the low-bit formats;
        # the 4- to 6-bit ones' experts, with larger weights, outweigh it
        t = _F16 if c["gate_up"] not in ("q4_K", "q5_K") and _dense_f16(c["shared"], c["tokens"]) else {"rel": 1e-5}
    return dict(t)


# ------------------------------------------------------------------------------ the same in 64 bits

# The lattices of the IQ formats: entries of 8 values from 8, 25, 43 (2 bits each) and of 4 values from 8 levels (3 bits
# each), an entry in a little-endian 16-bit word, base64.
_IQ2_XXS = (
    "AAACAAUACAAKABEAFAAgACIAKAAqAEEARABQAFgAYQBkAIAAggCKAKIAAQEEARABFQFAAYQBmAEAAgICIgKCAgEEBAQQBCEEJARABEIESARgBIEE"
    "hASQBKQEAAUCBQgFIAVGBWkFgAWRBQkGEAZABoQGpAYACAUICAgUCCgIQQhECFAIUgiICAQJQAkCChQKARAEEBAQIRBAEGAQhBCQEJUQABEIESAR"
    "UBFaEYARJBJFEgAUCBQgFCUUSRSAFBgVYhUAFhYWARgEGBAYQBiBGAAZBRmgGVEaACACIAogRCBhIIAggiApIUghACICIgEkBCQQJEAkViQAJUEl"
    "ZCWQJggoICiUKEQqAUAEQBBAGEAhQCRAQEBIQFZAYECBQIRAkEAAQSBBYUGAQYVBAUIQQkhCVkJoQgBECEQgRIBEmUQSRSRFAEYBSARIEEhASEVI"
    "AElYSWFJgklFSpBKAFAIUBFQGVAgUIBQiFAEUUJRpFGRUpBUklQKVQFWVFYAWBFYGVhkWEBZCFoEYBBgQGBoYABhVWEYYmBiAGQFZBBlEmWEZUJo"
    "AIACgAqAQYCCgASBGIFAgRGCAYQEhBCEFYRAhGCEAIVGhZSFCYZAhmCGAogEiRGKBJAQkCSQQJChkBaRgJFFkgCUIpRElFGVgZggmQKgUKCFoAmh"
    "AKIYpFCoBKk=")

_IQ2_S = (
    "AAACAAUACAAKABEAFAAWABkAIAAiACUAKABBAEQARgBJAFAAUgBVAFgAYQBkAGYAaQCAAIIAhQCIAJEAlACgAKUAqgABAQQBBgEJARABEgEVARgB"
    "IQEkAUABQgFFAUgBUQFUAVYBWQFgAWUBaAGBAYQBkAGSAZUBoQGkAQACAgIFAggCEQIUAiACKgJBAkQCRgJJAlACVQKAAoUCigKUAqICAQQEBAYE"
    "CQQQBBIEFQQYBCEEJAQmBCkEQARCBEUESARKBFEEVARWBFkEYARiBGUEgQSEBIYEiQSQBJUEmAShBKQEAAUCBQUFCAUKBREFFAUWBRkFIAUlBSgF"
    "QQVEBUYFSQVQBVIFVQVYBWEFZAWABYIFhQWIBZEFlAWgBQEGBAYGBgkGEAYVBkAGRQZIBlEGVAZgBoEGhAaQBgAIAggFCAgIEQgUCBYIGQggCCUI"
    "KghBCEQIRghJCFAIUghVCFgIYQhkCIAIhQiUCKoIAQkECRAJEgkVCRgJIQlACUUJSAlRCVQJYAmBCZAJAAoRChQKIgooCioKUAqZCgEQBBAGEAkQ"
    "EBASEBUQGBAhECQQJhBAEEIQRRBIEFEQVBBWEFkQYBBiEGUQaBCBEIQQhhCQEJUQmBChEKQQABECEQURCBEKERERFBEWERkRIBEiESURKBFBEUQR"
    "RhFJEVARUhFVEVgRYRFkEYARghGFEYgRkRGUEQESBBIJEhASFRIhEiQSQBJFElESVBKBEoQSkBIAFAIUBRQIFBEUFBQWFBkUIBQlFCgUQRREFEYU"
    "SRRQFFIUVRRYFGEUZBSAFIIUhRSIFJEUlBSgFAEVBBUGFQkVEBUSFRUVGBUhFSQVQBVCFUUVSBVRFVQVYBWBFYQVkBUAFgUWCBYRFhQWIBZBFkQW"
    "UBaAFqoWARgEGAYYCRgQGBUYGBghGEAYQhhFGEgYURhUGGAYgRiEGAAZAhkFGQgZERkUGSAZQRlEGVAZaRmiGQQaEBpAGlYaACACIAUgCCARIBQg"
    "FiAZICAgJSAqIEEgRCBQIFIgVSBkIIAgiiCUIKogASEEIRAhEiEVISEhQCFCIUUhUSFUIWAhgSGEIZAhACIKIiIiKCIqIkQiUCKIIooiqCIBJAQk"
    "BiQJJBAkFSQYJCEkJCRAJEIkRSRIJFEkVCRgJIEkhCSQJAAlBSUIJRElFCUgJUElRCVQJWYlgCUBJgQmECZAJlkmACgFKBEoFChBKEQoUCiKKKoo"
    "ASkEKRAplSkKKiIqZCqIKooqAUAEQAZACUAQQBJAFUAYQBpAIUAkQCZAQEBCQEVASEBKQFFAVEBWQFlAYEBiQGVAgUCEQJBAlUCYQKFApEAAQQJB"
    "BUEIQRFBFEEWQRlBIEEiQSVBQUFEQUZBSUFQQVJBVUFYQWFBZEGAQYJBhUGIQZFBlEGgQQFCBEIQQhJCFUIYQiRCQEJFQkhCUUJUQmBCgUKEQgBE"
    "AkQFRAhECkQRRBREFkQZRCBEIkQlRChEQUREREZESURQRFJEVURYRGFEZESARIJEhUSIRJFElESgRAFFBEUGRQlFEEUSRRVFGEUhRSRFQEVCRUVF"
    "SEVRRVRFYEVqRYFFhEWQRQBGAkYFRghGEUYURiBGQUZERlBGgEalRgFIBEgJSBBIEkgVSBhIIUgkSEBIQkhFSEhIUUhUSGBIhEiQSABJAkkFSQhJ"
    "EUkUSSBJQUlESVBJgEmWSQFKBEoQSkBKAFACUAVQCFARUBRQFlAZUCBQIlAlUChQQVBEUEZQSVBQUFJQVVBYUGFQZFCAUIJQhVCIUJFQlFABUQRR"
    "BlEJURBRElEVURhRIVEkUUBRQlFFUUhRUVFUUWBRgVGEUZBRAFIFUghSEVIUUiBSQVJEUlBSaVKAUgFUBFQGVAlUEFQSVBVUGFQhVCRUQFRCVEVU"
    "SFRRVFRUYFSBVIRUkFQAVQJVBVUIVRFVFFUgVUFVRFVQVYBVAVYEVhBWJlZAVgBYAlgFWAhYEVgUWCBYQVhEWFBYWliAWAFZBFkQWUBZAFoZWoVa"
    "qFoBYARgBmAQYBJgFWAYYCFgJGBAYEVgSGBRYFRgYGCEYJBgAGECYQVhCGERYRRhIGFBYURhUGGAYZlhBGIQYkBiVmKhYgBkBWQIZBFkFGQgZEFk"
    "RGRQZIBkAWUEZRBlQGVKZWhlkmUAZpRmAWgEaBBoZWiYaABpKmlCaqFqAIACgAWACIARgBSAGYAggCWAQYBEgFCAUoBVgFiAYYCAgIWAkYCUgAGB"
    "BIEJgRCBEoEVgRiBIYEkgUCBQoFFgUiBUYFUgYGBhIGQgamBAIIFggqCEYIUgkGCRIJQggGEBIQGhAmEEIQShBWEGIQhhECEQoRFhEiEUYRUhGCE"
    "gYSEhJCEAIUChQWFCIURhRSFIIVBhUSFUIWAhYqFAYYEhhCGKYZAhgCIBYgRiBSIQYhEiFCIoogBiQSJQIlliSKKWIpaioKKoooBkASQCZAQkBKQ"
    "FZAYkCSQQJBCkEWQSJBRkFSQYJCBkISQkJAAkQWREZEUkUGRRJFQkVqRAZIEkhCSQJKmkgCUApQFlAiUEZQUlCCUQZRElFCUgJSWlAGVBJUQlUCV"
    "mJWhlQCWRpZklgGYBJgQmCaYQJipmACZSZlSmZCaAKAFoAqgFKAioCqgQaBEoFCgoqCqoEChZaECogqiIqIooiqigqKIooqiqKIBpASkEKRApImk"
    "pKQApRmlUaYKqCiooqhUqYapCKoKqiCqIqooqoiqqqo=")

_IQ3_S = (
    "AAABAAIABQAHAAgACQAKAAwADgAQABEAFQAbACAAIgAlACcAKQArADAAMgA5ADwAPwBAAEEAQgBEAEgASQBNAFAAUwBXAFkAXQBkAHEAdQB6AIAA"
    "gQCFAIcAiACLAI4AkQCVAJgAnACiAKUApwCpAKsAuAC7AMMAyQDNANAA0gDZANsA3gDkAOgA6gD3APkA/QAAAQsBDwERARQBGgEgASMBKQE4AUIB"
    "RAFQAVIBVgFbAWEBZQFnAXYBewGGAYkBiwGZAaoBuQHAAcIBxAHQAdIB1gHbAegB7AEAAgECAgIEAggCCQILAg0CDwIQAhICGQIcAh4CLAIuAjEC"
    "OgJAAkECQwJGAkgCTAJRAlgCWwJhAmgCagJ4An4CgAKKAo0CjwKQApQCmgKgAqMCrQKwAroCwQLEAscCyALLAtEC1wLYAtwC4QLyAvgCAwMFAwoD"
    "DAMZAxsDIgMmAygDLANBA0gDSwNRA1gDWgNpA5ADlAOXA6QDpgPBA8MDyAPKA9ED3QPhA/ID+AMABAEEAwQFBAcECAQKBAwEDgQRBBMEFwQYBBoE"
    "IQQjBCUEKAQqBDcEOAQ7BD0EQARCBEgESwRPBFIEVQRZBFwEYgRpBIEEhASHBJEEkwSYBJ8EoQSrBK8EuQS8BMAEwgTFBMkE0gTUBNkE2wTiBOgE"
    "9gQBBQcFEAUTBRoFHQUhBToFPQVEBUkFUgVfBWAFawV4BYAFggWHBZEFrQWxBcUFyQXWBdgF4wXoBQIGCQYLBg0GDwYSBhkGGwYdBiIGJAYnBikG"
    "MwY5BkEGQwZFBkwGUQZTBmAGcAZ6Bn4GgAaKBpAGmgacBqgGwQbIBswG0QbTBtcG2AbhBuMG5wbtBvsGAwcJBw4HEgcZByoHMAc0B0EHSAdKB1UH"
    "WgdkB24HeweOB6EHwQfDB9AH0gfdBwAIBAgKCBAIFAgXCBoIIQgoCDgIQghHCEkISwhSCFgIXQhjCGkIbQiBCIMIiAiNCJEImwigCK8Isgi4CMQI"
    "yQjLCNAI0gjZCN0IAAkCCRQJHwkgCTkJRQlHCVEJcgmLCZwJsAnICc0J2AnjCekJAgoICgwKEgogCiQKJwoqCjYKPApBCkMKRQpKClEKWgp6CoAK"
    "iQqTCpgKngqrCsIKxwrICtcK5ArpCvUK+woBCwQLEAsaCyYLSgtWC2kLawuiC8ILxAvSCwkMCwwNDBkMGwwwDEAMUAxXDHQMigycDKIMrQyyDLgM"
    "wAzMDNEM4AwVDSMNMg1ADUMNXA1wDYUNoA3JDcsNAA4EDgcOEA4SDh4OIA4sDjIOQg5JDlQOYw5lDoEOhA6IDo4OkQ6YDqkOwg7aDt0O6w4BDwUP"
    "Cw8QDygPUg9iD4IPmQ/ADw==")

_IQ3_XXS = (
    "AAACAAQACQALAA8AEAASABkAIgA7AD0AQQBDAEgASgBRAFUAWABaAGEAbAB4AIAAggCEAIkAkACSAJkAmwCfAKkArwC9AMEAxwDIAMoA1QD4AAsB"
    "HwEkAS8BOwE9AUEBRwFaAWoBnQG0AcgBzAHOAeMB8QEBAgMCCAIKAhECEwIYAhoCHAInAigCQAJCAkkCUAJSAoECgwKIAooCkQKYAroCwALCAtAC"
    "2QLmAvYCAQMFAygDUANUA2YDeQOFA9ID4AMABAIECQQLBBAEEgQWBBkEIgRBBEMERQRIBEoEUQRYBHMEdwR4BIAEggSJBI8EkASSBJ8EoAStBMEE"
    "yATMBPgE/AQdBSsFQwVXBWEFfAXBBcMFzgXlBQEGCAYKBhEGEwYoBjUGOgZABkIGUAZZBmQGZgaBBoMGiAaVBqoGugbJBtsGGAcnBzoHQAdGB1IH"
    "bQeMB54HswfbB/AHBAgPCB0IHwgrCC8IfAiQCJ8IoAiwCLYIxwjlCAQJKQk0CVUJYwl4CcUJyAnKCdgJCgohCjgKQApGClYKbQqMCpoKugrCCusK"
    "CAsTCxcLOgtCC1kLqAvUC+ILFAwkDCYMNAxRDHEMjwy0DNgM3gwkDUUNag2bDcMN0Q0DDgUOBw4IDhoOKg5WDmAOig6lDqoOwA7NDtsO8A4RDyEP"
    "QA9CD1QPmA8=")

_TABLES = {}


def _table(name):
    if name not in _TABLES:
        text, levels, n = {"iq2_xxs": (_IQ2_XXS, [8, 25, 43], 8), "iq2_s": (_IQ2_S, [8, 25, 43], 8), "iq3_s": (_IQ3_S, list(range(1, 16, 2)), 4),
                           "iq3_xxs": (_IQ3_XXS, [4, 12, 20, 28, 36, 44, 52, 62], 4)}[name]
        v = np.frombuffer(base64.b64decode(text), dtype="<u2").astype(np.int64)
        bits = 2 if n == 8 else 3
        idx = (v[:, None] >> (bits * np.arange(n))) & ((1 << bits) - 1)
        _TABLES[name] = torch.from_numpy(np.array(levels, dtype=np.float64)[idx])
    return _TABLES[name]


_LEVELS4 = [-127., -104., -83., -65., -49., -35., -22., -10., 1., 13., 25., 38., 53., 69., 89., 113.]
_E2M1 = [0., .5, 1., 1.5, 2., 3., 4., 6., 0., -.5, -1., -1.5, -2., -3., -4., -6.]


def _f16(b):
    return b.contiguous().view(torch.float16).to(torch.float64)  # (blocks, 1)


def _bits(v, n, step=1):
    """(..., m) integers to (..., m, n): fields of `step` bits, the lowest first."""
    return (v[..., None] >> (step * torch.arange(n, device=v.device))) & ((1 << step) - 1)


def _signs(v7):
    """(..., m) 7-bit sign indices to (..., m, 8) factors: the 8th bit makes their count even."""
    s = _bits(v7, 7)
    s = torch.cat([s, s.sum(-1, keepdim=True) & 1], -1)
    return 1.0 - 2.0 * s.to(torch.float64)


def _words(b):
    """(blocks, 4m) bytes to (blocks, m) 32-bit words."""
    q = b.reshape(b.shape[0], -1, 4).long()
    return q[..., 0] | q[..., 1] << 8 | q[..., 2] << 16 | q[..., 3] << 24


def _k4_scales(b):
    """The 8 six-bit scales and minima of the 12 bytes of a Q4_K or Q5_K block."""
    b = b.long()
    lo, mid, hi = b[:, 0:4], b[:, 4:8], b[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | (lo >> 6 << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | (mid >> 6 << 4)], 1)
    return sc.double(), mn.double()


def _dequantize(dtype, raw):
    """GGUF blocks (flat bytes) to their weights in 64 bits."""
    b = raw.reshape(-1, F.type_size(dtype))
    nb, dev = b.shape[0], b.device
    if dtype == F.Q8_0:
        return (_f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    if dtype == F.MXFP4:
        q = torch.tensor(_E2M1, dtype=torch.float64, device=dev)[torch.cat([b[:, 1:] & 15, b[:, 1:] >> 4], 1).long()]
        return (q * torch.exp2(b[:, :1].double() - 127)).reshape(-1)
    if dtype in (F.Q4_K, F.Q5_K):
        sc, mn = _k4_scales(b[:, 4:16])
        qs = b[:, 16:144] if dtype == F.Q4_K else b[:, 48:176]
        q = _bits(qs.reshape(nb, 4, 32).long(), 2, 4).transpose(2, 3).reshape(nb, 8, 32)
        if dtype == F.Q5_K:
            q = q + 16 * _bits(b[:, 16:48].long(), 8).transpose(1, 2)
        return ((_f16(b[:, :2]) * sc)[..., None] * q - (_f16(b[:, 2:4]) * mn)[..., None]).reshape(-1)
    if dtype == F.Q2_K:
        sc = b[:, :16].long()
        q = _bits(b[:, 16:80].reshape(nb, 2, 32).long(), 4, 2).transpose(2, 3).reshape(nb, 16, 16)
        return ((_f16(b[:, 80:82]) * (sc & 15))[..., None] * q - (_f16(b[:, 82:84]) * (sc >> 4))[..., None]).reshape(-1)
    if dtype == F.Q6_K:
        lo = _bits(b[:, :128].reshape(nb, 2, 2, 32).long(), 2, 4).permute(0, 1, 4, 2, 3).reshape(nb, 2, 4, 32)
        hi = _bits(b[:, 128:192].reshape(nb, 2, 32).long(), 4, 2).transpose(2, 3)
        q = (lo + 16 * hi - 32).reshape(nb, 16, 16)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return ((_f16(b[:, 208:210]) * sc)[..., None] * q).reshape(-1)
    if dtype == F.IQ2_XXS:
        w = _words(b[:, 2:66]).reshape(nb, 8, 2)
        g = _table("iq2_xxs").to(dev)[_bits(w[..., 0], 4, 8)]
        dl = _f16(b[:, :2]) * (0.5 + (w[..., 1] >> 28)) * 0.25
        return (dl[..., None, None] * g * _signs(_bits(w[..., 1], 4, 7))).reshape(-1)
    if dtype == F.IQ2_S:
        i = b[:, 2:34].long() | _bits(b[:, 66:74].long(), 4, 2).reshape(nb, 32) << 8
        s = 1.0 - 2.0 * _bits(b[:, 34:66].long(), 8).double()
        dl = (_f16(b[:, :2]) * (0.5 + _bits(b[:, 74:82].long(), 2, 4).reshape(nb, 16)) * 0.25).repeat_interleave(2, 1)
        return (dl[..., None] * _table("iq2_s").to(dev)[i] * s).reshape(-1)
    if dtype == F.IQ3_S:
        i = b[:, 2:66].long() | _bits(b[:, 66:74].long(), 8).reshape(nb, 64) << 8
        s = 1.0 - 2.0 * _bits(b[:, 74:106].long(), 8).double().reshape(nb, 64, 4)
        dl = (_f16(b[:, :2]) * (1 + 2 * _bits(b[:, 106:110].long(), 2, 4).reshape(nb, 8))).repeat_interleave(8, 1)
        return (dl[..., None] * _table("iq3_s").to(dev)[i] * s).reshape(-1)
    if dtype == F.IQ3_XXS:
        g = _table("iq3_xxs").to(dev)[b[:, 2:66].long()].reshape(nb, 8, 4, 8)
        w = _words(b[:, 66:98])
        dl = _f16(b[:, :2]) * (0.5 + (w >> 28)) * 0.5
        return (dl[..., None, None] * g * _signs(_bits(w, 4, 7))).reshape(-1)
    if dtype == F.IQ4_XS:
        high = b[:, 2:3].long() | b[:, 3:4].long() << 8
        ls = _bits(b[:, 4:8].long(), 2, 4).reshape(nb, 8) | _bits(high, 8, 2).reshape(nb, 8) << 4
        q = _bits(b[:, 8:136].reshape(nb, 8, 16).long(), 2, 4).transpose(2, 3).reshape(nb, 8, 32)
        v = torch.tensor(_LEVELS4, dtype=torch.float64, device=dev)[q]
        return ((_f16(b[:, :2]) * (ls - 32))[..., None] * v).reshape(-1)
    raise ValueError(F.NAMES[dtype])


def _matrix(dtype, raw, shape):
    return _dequantize(dtype, raw).reshape(shape)


def _silu_mul(g, u):
    return g * torch.sigmoid(g) * u


def _exact_layer(c, d):
    x = d["x"].double()
    logits = d["logits"].double() if "logits" in d else x @ d["router"].double().t()
    p, ids = torch.sort(torch.softmax(logits, 1), dim=1, descending=True, stable=True)
    p, ids = p[:, :c["top_k"]], ids[:, :c["top_k"]]
    w = p / p.sum(1, keepdim=True)
    out = torch.zeros_like(x)
    slot_of = {e: s for s, e in enumerate(d["resident"].tolist())} if d["resident"] is not None else None
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        s = slot_of[e] if slot_of is not None else e
        m = []
        for raw, dt, shape in zip(d["raw"], d["dtypes"], d["shapes"]):
            size = F.matrix_bytes(dt, *shape)
            m.append(_matrix(dt, raw[s * size:(s + 1) * size], shape))
        g, u = x[t] @ m[0].t(), x[t] @ m[1].t()
        if d["bias"] is not None:
            g, u = (g + d["bias"][0][e].double()).clamp(max=7.0), (u + d["bias"][1][e].double()).clamp(-7.0, 7.0)
            y = ((u + 1) * g * torch.sigmoid(1.702 * g)) @ m[2].t() + d["bias"][2][e].double()
        else:
            y = _silu_mul(g, u) @ m[2].t()
        out.index_add_(0, t, w[t, j][:, None] * y)
    if c["kind"] == "block":
        g, u, dn = [_matrix(dt, raw, shape) for raw, dt, shape in d["shared"]]
        y = _silu_mul(x @ g.t(), x @ u.t()) @ dn.t()
        return out + y * torch.sigmoid(x @ d["gate_inp"].double())[:, None], None, w, logits
    return out, None, w


def exact(case, seed):
    gen = _gen(seed)
    if case["kind"] == "shrink":
        return None  # bytes: no value in 64 bits
    if case["kind"] == "dense":
        dt, shape = F.BY_NAME[case["weight"]], (case["n"], case["k"])
        return [x.double() @ _matrix(dt, raw, shape).t() for raw, x in _dense_inputs(case, gen)]
    return [_exact_layer(case, d) for d in _moe_inputs(case, gen)]
