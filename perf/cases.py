"""The work that a program has this framework do, as cases that can be timed: one pass of one MoE MLP layer.

A case is one layer (experts, sizes, formats), one batch of tokens and one entry point:

  layer   `MxMoELayer(...)(hidden, topk_ids, topk_weights)`: a serving engine's fused-MoE call after its own routing
  logits  `MxMoELayer.forward_from_logits`: the same with the routing (softmax, top-k, renormalisation) inside
  graph   `MxMoELayer.capture(...)`: inputs copied into the static tensors, then `replay()`: a decode loop
  ops     the operators of `mxmoe_amd.ops` one after the other, the sequence that callers of the original `mxmoe_ops` run
  gemm    the two GroupGEMM launches alone over permuted, quantised rows in memory: what `bench.py` calls a step

The layers are those of `mxmoe_amd.synth.CONFIGS` (Qwen1.5-MoE, DeepSeek-V2-Lite, Mixtral-8x7B), with Qwen's shared expert where the case
has one.  Every state has weights of its own, as every layer of a model has, so no pass finds them in a cache.
"""
from __future__ import annotations

import math

import torch

from mxmoe_amd import ops, synth
from mxmoe_amd.layer import MxMoELayer

W8A16 = (16, 8, 128, False)
# name -> (formats, share of each, w8a8 blocks in fp8): the mixes a bit-width allocation hands out
MIXES = {
    "fp16": ((synth.FP16,), (1.0,), False),
    "w4a4": ((synth.W4A4,), (1.0,), False),
    "w4a4/w8a8": ((synth.W4A4, synth.W8A8), (0.5, 0.5), False),
    "w4a16/w3a16": ((synth.W4A16, synth.W3A16), (0.7, 0.3), False),
    "w4a16": ((synth.W4A16,), (1.0,), False),
    "w8a16/w2a16": ((W8A16, synth.W2A16), (0.5, 0.5), False),
    "w4a4/w8a8/w4a16": ((synth.W4A4, synth.W8A8, synth.W4A16), (0.4, 0.4, 0.2), False),
    "w4a4g128/fp8/w8a16/w2a16": ((synth.W4A4G128, synth.W8A8, W8A16, synth.W2A16), (0.3, 0.3, 0.2, 0.2), True),
    "w4a4/fp8": ((synth.W4A4, synth.W8A8), (0.5, 0.5), True),
}
# experts, top-k, hidden, intermediate, shared experts
QWEN = dict(experts=60, topk=4, hidden=2048, inter=1408, shared=0)
QWEN_SHARED = dict(QWEN, shared=4)
DS2 = dict(experts=64, topk=6, hidden=2048, inter=1408, shared=2)
MIXTRAL = dict(experts=8, topk=2, hidden=4096, inter=14336, shared=0)


def listed():
    return [
        # one sequence decoding: a handful of experts, one row each; latency and launches
        dict(name="decode 1", entry="layer", **DS2, tokens=1, mix="w4a16/w3a16", routing="gaussian"),
        # a decode batch of the same layer, every expert a few rows: the weights' bytes
        dict(name="decode 32", entry="layer", **DS2, tokens=32, mix="w4a16/w3a16", routing="gaussian"),
        # a decode loop on a captured graph, quantised activations with the online rotation
        dict(name="decode 8 graph", entry="graph", **QWEN, tokens=8, mix="w4a4/w8a8", routing="gaussian"),
        # a decode batch from the router's logits, skewed experts, with the shared expert
        dict(name="decode 64 logits", entry="logits", **QWEN_SHARED, tokens=64, mix="w4a4/w8a8", routing="zipf"),
        # few, large experts in a small batch: over a gigabyte of weights
        dict(name="decode 16 large", entry="layer", **MIXTRAL, tokens=16, mix="w4a4/w8a8/w4a16", routing="biased"),
        # a short prompt or a speculative batch of odd length: weight-only experts with some tens of rows
        dict(name="chunk 201", entry="layer", **DS2, tokens=201, mix="w4a16/w3a16", routing="gaussian"),
        # a chunk of a prefill, no quantisation
        dict(name="chunk 512 fp16", entry="layer", **QWEN, tokens=512, mix="fp16", routing="gaussian"),
        # the operators in sequence on a chunk of odd length
        dict(name="ops 777", entry="ops", **QWEN, tokens=777, mix="w4a4/w8a8", routing="zipf"),
        # a chunked prefill over the less usual formats, next to each other in one launch
        dict(name="chunk 2049 formats", entry="layer", **DS2, tokens=2049, mix="w4a4g128/fp8/w8a16/w2a16", routing="gaussian"),
        # a full prefill batch, uniform 4-bit operands
        dict(name="prefill 8192", entry="layer", **QWEN, tokens=8192, mix="w4a4", routing="gaussian"),
        # the headline benchmark's step: both launches on skewed experts
        dict(name="gemm 8192", entry="gemm", **QWEN, tokens=8192, mix="w4a4/w8a8", routing="zipf"),
        # a full prefill batch on large experts in three formats
        dict(name="prefill 8192 large", entry="layer", **MIXTRAL, tokens=8192, mix="w4a4/w8a8/w4a16", routing="biased"),
    ]


def draw(rng):
    shape = rng.choice([QWEN, QWEN_SHARED, DS2, DS2, MIXTRAL])
    mix = rng.choice(list(MIXES))
    entry = rng.choice(["layer", "layer", "layer", "logits", "graph", "ops", "gemm"])
    most = 8192
    if entry == "graph":
        most = 256  # decode loops
    elif entry == "ops":
        most = 4096
    if shape is MIXTRAL and mix not in ("w4a4", "w4a4/w8a8", "w4a4/w8a8/w4a16"):
        most = min(most, 2048)  # formats of fewer operations a second: no more work than the largest listed case
    tokens = int(math.exp(rng.uniform(0.0, math.log(most + 1))))
    return dict(entry=entry, **shape, tokens=max(1, min(most, tokens)), mix=mix, routing=rng.choice(["gaussian", "zipf", "biased"]))


def _config(case) -> synth.MoEConfig:
    formats, probs, _ = MIXES[case["mix"]]
    return synth.MoEConfig("case", "case", case["experts"], case["topk"], case["hidden"], case["inter"], case["tokens"], num_shared=case["shared"],
                           routing=case["routing"], formats=formats, format_probs=probs, rotate=1)


class _Weights:
    """fp16 N(0, 0.02) weights of expert e, made when the layer asks for them."""

    def __init__(self, cfg, gen):
        self.cfg, self.gen = cfg, gen

    def __getitem__(self, e):
        c = self.cfg
        i = c.inter * (c.num_shared if e == c.num_experts else 1)

        def w(n, k):
            return torch.randn(n, k, generator=self.gen, device="cuda", dtype=torch.float16).mul_(0.02)

        return w(2 * i, c.hidden), w(c.hidden, i)


def _logits(case, gen):
    t, e = case["tokens"], case["experts"]
    if case["routing"] == "zipf":  # expert popularity ~ rank^-1.2, every token draws distinct experts
        p = torch.arange(1, e + 1, device="cuda", dtype=torch.float32) ** -1.2
        u = torch.rand(t, e, generator=gen, device="cuda").clamp_(1e-20, 1.0)
        return (p / p.sum()).log() - (-u.log()).clamp_min(1e-20).log()
    z = torch.randn(t, e, generator=gen, device="cuda")
    if case["routing"] == "biased":
        z = z + 0.5 * torch.randn(e, generator=gen, device="cuda")
    return z


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    cfg = _config(case)
    layer = MxMoELayer(cfg, weights=_Weights(cfg, gen), fp8=MIXES[case["mix"]][2])
    s = {"case": case, "cfg": cfg, "layer": layer, "hidden": torch.randn(cfg.tokens, cfg.hidden, generator=gen, device="cuda", dtype=torch.float16)}
    logits = _logits(case, gen)
    w, ids = torch.topk(torch.softmax(logits, dim=1), cfg.topk, dim=-1)
    s["ids"], s["w"] = ids.to(torch.int32), (w / w.sum(dim=-1, keepdim=True)).contiguous()
    if case["entry"] == "logits":
        s["logits"] = logits
    elif case["entry"] == "graph":
        s["captured"] = layer.capture(cfg.tokens)
    elif case["entry"] == "ops":
        s["w13"], s["s13"] = [p.data for p in layer.w13], [p.scale for p in layer.w13]
        s["w2"], s["s2"] = [p.data for p in layer.w2], [p.scale for p in layer.w2]
    elif case["entry"] == "gemm":
        layer.prepare(s["hidden"], s["ids"])
        layer.gate_up()
        layer.act()
    return s


def _run_ops(s):
    cfg, layer = s["cfg"], s["layer"]
    e, k, i, sh = cfg.num_experts, cfg.hidden, cfg.inter, cfg.num_shared
    i_sh = i * max(sh, 1)
    inp, sa, mid, _, _, mid_store, recv, _, dst = ops.quant_inp_act(s["hidden"], s["ids"], e, i, sh, layer.qp_gate_up, rotate=cfg.rotate, fp8=layer.fp8)
    ops.gg_mxmoe_share_fused(inp, s["w13"], sa, s["s13"], mid, 2 * i, k, 2 * i_sh, k, layer.qp_gate_up, recv, kernel_id=layer.kid_gate_up)
    inp2, sa2, out, _, _, out_store = ops.silu_mul_then_quant(mid_store, len(mid), e, k, i, sh, cfg.tokens, cfg.topk, dst, recv, layer.qp_down,
                                                              rotate=cfg.rotate, fp8=layer.fp8)
    ops.gg_mxmoe_share_fused(inp2, s["w2"], sa2, s["s2"], out, k, i, k, i_sh, layer.qp_down, recv, kernel_id=layer.kid_down)
    return ops.gg_unpermute_out(out_store, s["ids"], s["w"], e, k, sh)


def run(s):
    entry, layer = s["case"]["entry"], s["layer"]
    if entry == "layer":
        return layer(s["hidden"], s["ids"], s["w"])
    if entry == "logits":
        return layer.forward_from_logits(s["hidden"], s["logits"], renormalise=True)
    if entry == "graph":
        c = s["captured"]
        c.hidden.copy_(s["hidden"])
        c.topk_ids.copy_(s["ids"])
        c.topk_weights.copy_(s["w"])
        return c.replay()
    if entry == "ops":
        return _run_ops(s)
    layer.gate_up()
    layer.down()
    cfg, st = s["cfg"], layer.state
    rows, shared = cfg.tokens * cfg.topk, cfg.tokens * (cfg.num_shared > 0)
    # (the stores are sized for more rows than a layer produces: what the launches wrote)
    return {"mid": st["mid_store"][:2 * cfg.inter * (rows + shared * cfg.num_shared)], "out": st["out_store"][:cfg.hidden * (rows + shared)]}


def _block_bytes(n, k, q):
    """Packed weights and scales of one [n, k] block."""
    a, w, g, _ = q
    if w >= 16:
        return 2 * n * k
    return n * k * w // 8 + (4 if a >= 16 else 2) * n * (k // g if g > 0 else 1)


def work(case):
    """Each weight of an expert that gets tokens read once, the tokens in, the tokens out (`gemm`: the packed rows in, both outputs)."""
    cfg = _config(case)
    t, e, k, i = cfg.tokens, cfg.num_experts, cfg.hidden, cfg.inter
    rows = t * cfg.topk
    i_sh = i * cfg.num_shared
    formats = synth.draw_formats(cfg)
    hit = 1.0 - (1.0 - cfg.topk / e) ** t  # share of the experts that a batch reaches
    weights = hit * sum(_block_bytes(2 * i, k, gu) + _block_bytes(k, i, dn) for gu, dn in formats[:e])
    if i_sh:
        weights += _block_bytes(2 * i_sh, k, formats[e][0]) + _block_bytes(k, i_sh, formats[e][1])
    flops = 6 * k * (rows * i + t * i_sh)
    if case["entry"] == "gemm":
        bits = [sum(min(f[b][0], 16) for f in formats[:e]) / e for b in (0, 1)]
        act = rows * (k * bits[0] + i * bits[1]) / 8 + (t * (k * min(formats[e][0][0], 16) + i_sh * min(formats[e][1][0], 16)) / 8 if i_sh else 0)
        out = 2 * rows * (2 * i + k) + (2 * t * (2 * i_sh + k) if i_sh else 0)
        return {"bytes": weights + act + out, "flops": flops}
    return {"bytes": weights + 4 * t * k + rows * 8, "flops": flops}


def tolerance(case):
    """fp16 operands, intermediate rows and outputs with fp32 sums; quantised intermediate rows turn a last-bit difference of a value
    on the edge of two codes into a whole code of 4 bits."""
    if all(f[0] >= 16 for f in MIXES[case["mix"]][0]):
        return {"rel": 2e-3}
    return {"rel": 1e-2}
