"""Timed cases of the fused-MoE path, through its public entry points.

A case is one MoE layer call (or the loose steps around it) as an inference
engine makes it: router logits to experts, the fused layer in each weight
format, the reference-signature call on its routing tuple, the biased swiglu
layer, the SGLang adapter, and the separate operators a program uses that
runs its own expert GEMMs. Decode batches of one to a few dozen tokens and
prefill chunks of up to 8192 are both in, with hidden and intermediate sizes
that are any multiple of the granularity the layer accepts (128; int8: 256).
"""

import math
import os
import sys
from types import SimpleNamespace

import torch

_PKG = os.path.join(os.getcwd(), "flaggems-sglang_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import flaggems_sglang as fgs  # noqa: E402
from flaggems_sglang import quant  # noqa: E402


def _layer(name, entry, mode, m, hidden, inter, experts, topk, **more):
    case = dict(name=name, entry=entry, mode=mode, m=m, hidden=hidden, inter=inter,
                experts=experts, topk=topk, scoring="softmax", hot=0, scale=1.0,
                activation="silu", on_input=False)
    case.update(more)
    return case


def listed():
    return [
        # one token of a chat request on a fine-grained layer: the router and
        # the experts; launches and latency count
        _layer("decode_one", "router", "bf16", 1, 2048, 768, 128, 8),
        # a few concurrent requests on the biased swiglu layer
        _layer("decode_bias", "bias", "bf16", 7, 2944, 2944, 32, 4),
        # a decode batch on few large experts, through the SGLang adapter
        _layer("decode_bf16", "adapter", "bf16", 32, 4096, 14336, 8, 2),
        # decode batches on quantised experts, the router included; the fp8
        # layer scales its output as its model does
        _layer("decode_fp8", "router", "fp8", 37, 7168, 2048, 256, 8,
               scoring="sigmoid", scale=2.5),
        _layer("decode_int8", "router", "int8", 64, 3584, 2560, 64, 8),
        # prefill chunks: fine-grained experts with skewed load, an odd count
        _layer("prefill_skewed", "fused", "bf16", 1999, 2048, 768, 128, 8, hot=8),
        # few large experts
        _layer("prefill_bf16", "fused", "bf16", 4096, 4096, 14336, 8, 2),
        # quantised experts
        _layer("prefill_fp8", "fused", "fp8", 4096, 7168, 2048, 256, 8,
               scoring="sigmoid", scale=2.5),
        _layer("prefill_int8", "fused", "int8", 8192, 3584, 2560, 64, 8),
        # the biased swiglu layer: 2880-wide weights padded to the granularity
        _layer("prefill_bias", "bias", "bf16", 4096, 2944, 2944, 32, 4),
        # the reference's own benchmark shape and call: the routing tuple from
        # (weights, ids), then triton_kernel_fused_experts on it
        _layer("routed_call", "routed", "bf16", 1024, 1280, 3072, 64, 8),
        # a program with expert GEMMs of its own: router, alignment,
        # activation, requantisation, top-k sum
        _layer("loose_steps", "steps", "fp8", 2048, 7168, 2048, 256, 8, scoring="sigmoid"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        entry = rng.choice(["router", "fused", "fused", "adapter", "bias", "bias", "routed",
                            "steps"])
        mode = rng.choice(["bf16", "bf16", "fp8", "int8"]) if entry in ("router", "fused") else (
            "fp8" if entry == "steps" else "bf16")
        experts = rng.choice([8, 16, 32, 64, 128, 160, 256])
        topk = rng.choice([1, 2, 4, 6, 8])
        m = _log_int(rng, 1, 8192)
        step = 256 if mode == "int8" else 128
        hidden = step * _log_int(rng, 1024 // step, 7168 // step)
        inter = step * _log_int(rng, 256 // step, 14336 // step)
        more = dict(scoring=rng.choice(["softmax", "sigmoid"]), hot=rng.choice([0, 0, 4]),
                    scale=rng.choice([1.0, 1.0, 2.5]) if entry in ("router", "fused") else 1.0)
        if entry in ("fused", "adapter", "routed"):
            more["activation"] = rng.choice(["silu", "silu", "silu", "gelu"])
        if entry in ("fused", "bias"):
            more["on_input"] = rng.random() < 0.2
        case = _layer("", entry, mode, m, hidden, inter, experts, topk, **more)
        del case["name"]
        if entry == "steps":
            if m * topk * (3 * inter + hidden) > 4e8 or m < 16:
                continue
            return case
        # the largest drawn layer is no more work than the largest listed ones
        weights = 3.0 * experts * hidden * inter * (2 if mode == "bf16" else 1)
        flops = 6.0 * m * topk * hidden * inter
        if weights > 8e9 or flops > (0.7e12 if hidden % 256 else 2e12):
            continue
        return case


# ------------------------------------------------------------------ inputs ---
def _weights(case, gen):
    """Expert weights [E, 2N, K] and [E, K, N] (and their scales)."""
    e, k, n = case["experts"], case["hidden"], case["inter"]
    dev = "cuda"

    def one(rows, cols):
        w = torch.empty((e, rows, cols), dtype=torch.bfloat16, device=dev)
        w.normal_(0.0, 0.02, generator=gen)
        return w

    w1, s1 = one(2 * n, k), None
    if case["mode"] != "bf16":
        w1, s1 = _quantised(w1, case["mode"])
    w2, s2 = one(k, n), None
    if case["mode"] != "bf16":
        w2, s2 = _quantised(w2, case["mode"])
    return w1, w2, s1, s2


def _quantised(w, mode):
    return (quant.quantize_fp8_block if mode == "fp8" else quant.quantize_int8_channel)(w)


def _logits(case, gen):
    logits = torch.randn((case["m"], case["experts"]), generator=gen, device="cuda")
    if case["hot"]:
        # a few popular experts, spread over the id range
        step = max(1, case["experts"] // case["hot"])
        logits[:, step // 2::step] += 2.0
    return logits


def _scores(case, logits):
    return logits.softmax(-1) if case["scoring"] == "softmax" else logits.sigmoid()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    m, k, n, e, topk = (case[x] for x in ("m", "hidden", "inter", "experts", "topk"))
    s = SimpleNamespace(case=case)
    s.logits = _logits(case, gen)
    if case["entry"] == "steps":
        rows = m * topk
        s.gate_up = torch.empty((rows, 2 * n), dtype=torch.bfloat16, device="cuda")
        s.gate_up.normal_(generator=gen)
        s.y = torch.empty((m, topk, k), dtype=torch.bfloat16, device="cuda")
        s.y.normal_(generator=gen)
        return s
    s.x = torch.empty((m, k), dtype=torch.bfloat16, device="cuda")
    s.x.normal_(generator=gen)
    s.w1, s.w2, s.s1, s.s2 = _weights(case, gen)
    s.kw = {}
    if case["mode"] == "fp8":
        s.kw = dict(use_fp8_w8a8=True, block_shape=[128, 128], w1_scale=s.s1, w2_scale=s.s2)
    elif case["mode"] == "int8":
        s.kw = dict(use_int8_w8a8=True, per_channel_quant=True, w1_scale=s.s1, w2_scale=s.s2)
    if case["entry"] == "bias":
        s.b1 = 0.1 * torch.randn((e, 2 * n), generator=gen, device="cuda")
        s.b2 = 0.1 * torch.randn((e, k), generator=gen, device="cuda")
    if case["entry"] == "router":
        return s
    w, ids = torch.topk(_scores(case, s.logits), topk, dim=-1)
    s.ids = ids.to(torch.int32)
    s.w = (w / w.sum(-1, keepdim=True)).float()
    if case["entry"] == "adapter":
        config = SimpleNamespace(num_experts=e, activation=case["activation"],
                                 apply_router_weight_on_input=False, no_combine=False,
                                 routed_scaling_factor=case["scale"])
        s.runner = SimpleNamespace(runner=SimpleNamespace(config=config))
        s.layer = SimpleNamespace(w13_weight=s.w1, w2_weight=s.w2)
    elif case["entry"] == "routed":
        # the reference's layouts [E, K, 2N] and [E, N, K], as its plugin
        # passes them: transposed views of the native weights
        s.w1t, s.w2t = s.w1.transpose(-1, -2), s.w2.transpose(-1, -2)
    return s


def run(s):
    case = s.case
    entry, topk = case["entry"], case["topk"]
    scale = case["scale"] if case["scale"] != 1.0 else None
    if entry == "router":
        w, ids = fgs.fused_topk(s.x, s.logits, topk, scoring_func=case["scoring"])
        out = fgs.fused_moe(s.x, s.w1, s.w2, w, ids, routed_scaling_factor=scale, **s.kw)
        return {"out": out, "weights": w, "ids": ids}
    if entry == "fused":
        return fgs.fused_moe(s.x, s.w1, s.w2, s.w, s.ids, activation=case["activation"],
                             apply_router_weight_on_input=case["on_input"],
                             routed_scaling_factor=scale, **s.kw)
    if entry == "bias":
        return fgs.fused_moe_with_bias(
            s.x, s.w1, s.b1, s.w2, s.b2, s.w, s.ids,
            apply_router_weight_on_input=case["on_input"], gemm1_alpha=1.702,
            gemm1_clamp_limit=7.0, interleaved=False)
    if entry == "adapter":
        dispatch = SimpleNamespace(hidden_states=s.x, topk_output=SimpleNamespace(
            topk_weights=s.w, topk_ids=s.ids))
        return fgs.fused_moe_flagos(s.runner, s.layer, dispatch).hidden_states
    if entry == "routed":
        routing, gather, scatter = fgs.standard_topk_to_routing(s.w, s.ids, case["experts"])
        out = fgs.triton_kernel_fused_experts(s.x, s.w1t, s.w2t, routing, gather, scatter,
                                              activation=case["activation"])
        return {"out": out, "hist": routing.expt_hist, "gather": gather.src_indx}
    w, ids = fgs.fused_topk(s.y[:, 0], s.logits, topk, scoring_func=case["scoring"])
    order, blocks, padded = fgs.moe_align_block_size(ids, case["experts"], 64)
    act = fgs.silu_and_mul(s.gate_up)
    q, qs = fgs.per_token_group_quant_fp8(act)
    total = fgs.moe_sum(s.y)
    return {"weights": w, "ids": ids, "order": order, "blocks": blocks, "padded": padded,
            "act": act, "codes": q.view(torch.uint8), "scales": qs, "sum": total}


# ------------------------------------------------------ work and exactness ---
def work(case):
    m, k, n, e, topk = (case[x] for x in ("m", "hidden", "inter", "experts", "topk"))
    router = m * e * 4 + m * topk * 8
    if case["entry"] == "steps":
        rows = m * topk
        pairs = rows * (2 * n * 2 + n * 2 + n * 2 + n + n // 128 * 4)
        return {"bytes": router + rows * 8 + pairs + rows * k * 2 + m * k * 2, "flops": 0}
    touched = e * (1.0 - (1.0 - topk / e) ** m)  # experts some token picks
    per_expert = 3 * k * n * (2 if case["mode"] == "bf16" else 1)
    if case["mode"] == "fp8":
        per_expert += 3 * k * n // (128 * 128) * 4
    elif case["mode"] == "int8":
        per_expert += (2 * n + k) * 4
    if case["entry"] == "bias":
        per_expert += (2 * n + k) * 4
    total = touched * per_expert + 2 * m * k * 2 + m * topk * 8
    if case["entry"] == "router":
        total += router
    elif case["entry"] == "routed":
        total += m * topk * 20
    return {"bytes": int(total), "flops": 6 * m * topk * k * n}


def tolerance(case):
    # Three to four times the measured distance from the 64-bit result: 0.0017
    # for one rounding to bf16 (a code of the requantised activation moves
    # with it now and then), 0.0039 for the layer's bf16 gate, up, activation
    # and slot values; requantising the intermediate, where one bf16 step
    # moves a value to the next code, gives 0.012 in int8 and 0.018 in fp8
    # (of which 0.03 is as much as says anything).
    if case["entry"] == "steps":
        return {"rel": 7e-3, "max": 0.1, "differ": 2e-3}
    if case["mode"] != "bf16":
        return {"rel": 3e-2, "max": 0.4}
    return {"rel": 1.4e-2, "max": 0.2}


def _fp8_group(x):
    """1 x 128 group e4m3 codes' values in 64 bits."""
    g = x.float().reshape(x.shape[0], -1, 128)
    scale = g.abs().amax(-1, keepdim=True).clamp(min=1e-10) / 448.0
    q = (g / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.double() * scale.double()).reshape(x.shape)


def _int8_token(x):
    f = x.float()
    scale = f.abs().amax(-1, keepdim=True).clamp(min=1e-10) / 127.0
    return (f / scale).round().clamp(-127, 127).double() * scale.double()


def _dequantised(w, scale, mode):
    w = w.double()
    if mode == "fp8":
        w = w.reshape(w.shape[0] // 128, 128, w.shape[1] // 128, 128)
        w = (w * scale.double()[:, None, :, None]).reshape(w.shape[0] * 128, -1)
    elif mode == "int8":
        w = w * scale.double()[:, None]
    return w


def _top(scores, topk):
    # ranked by score, ties to the lower expert
    v, ids = torch.sort(scores, dim=-1, descending=True, stable=True)
    return v[:, :topk], ids[:, :topk]


def exact(case, seed):
    s = prepare(case, seed)
    m, k, n, e, topk = (case[x] for x in ("m", "hidden", "inter", "experts", "topk"))
    entry, mode = case["entry"], case["mode"]
    if entry in ("router", "steps"):
        _, ids = _top(s.logits, topk)
        w = _scores(case, s.logits.double()).gather(1, ids)
        w = w / w.sum(-1, keepdim=True)
    else:
        w, ids = s.w.double(), s.ids.long()
    if entry == "steps":
        gate, up = s.gate_up.double().chunk(2, dim=-1)
        return {"weights": w, "ids": None, "order": None, "blocks": None, "padded": None,
                "act": gate * torch.sigmoid(gate) * up, "codes": None, "scales": None,
                "sum": s.y.double().sum(1)}
    x = {"bf16": lambda t: t.double(), "fp8": _fp8_group, "int8": _int8_token}[mode]
    xq = x(s.x)
    out = torch.zeros((m, k), dtype=torch.float64, device="cuda")
    for j in range(e):
        tok, slot = torch.where(ids == j)
        if tok.numel() == 0:
            continue
        gamma = w[tok, slot][:, None]
        w1 = _dequantised(s.w1[j], None if s.s1 is None else s.s1[j], mode)
        h = xq[tok] @ w1.T
        del w1
        if entry == "bias":
            h = h + s.b1[j].double()
        gate, up = h.chunk(2, dim=-1)
        if case["on_input"] and entry != "bias":
            gate, up = gate * gamma, up * gamma
        if entry == "bias":
            gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
            act = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
            if case["on_input"]:
                act = act * gamma
        elif case["activation"] == "gelu":
            act = torch.nn.functional.gelu(gate) * up
        else:
            act = gate * torch.sigmoid(gate) * up
        if mode != "bf16":
            act = x(act)
        y = act @ _dequantised(s.w2[j], None if s.s2 is None else s.s2[j], mode).T
        if entry == "bias":
            y = y + s.b2[j].double()
        out.index_add_(0, tok, y if case["on_input"] else y * gamma)
    out = out * case["scale"]
    if entry == "router":
        return {"out": out, "weights": w, "ids": None}
    if entry == "routed":
        return {"out": out, "hist": None, "gather": None}
    return out
