"""The work that a user of this package has it do, as cases that can be timed: decode steps over a quantised
cache, the quantisers that fill the cache at prefill, and one attention layer taken from prompt to tokens.

A case is a dict of plain values.  `prepare` makes what a program holds before the call, `run` is one pass through
the public entry points, `work` the bytes and operations that pass cannot do without, `tolerance` how far two
correct implementations of it may lie apart.
"""
from __future__ import annotations

import math

import torch

from calibquant_amd import ops
from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
from calibquant_amd.patch_internvl import ATTN_FORWARD_FUNCTIONS

D = 128
CLIP_K = {1: 0.5, 2: 1.0}      # the clip factors the attention patch uses per bit width
CLIP_V = {1: 0.3, 2: 1.0}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _decode(name, batch, q_heads, kv_heads, tokens, rows, bits=1, dtype="bf16", values="channel", system=0, option="none"):
    """One decode-attention step of one layer.  `rows`: the full-precision window, of which `system` precede the
    image tokens.  `option`: "mask" (left-padded batch), "device-rows" (the window's length read on the device,
    as in a recorded step) or "none"."""
    return {"name": name, "kind": "decode", "batch": batch, "q_heads": q_heads, "kv_heads": kv_heads, "tokens": tokens,
            "rows": rows, "bits": bits, "dtype": dtype, "values": values, "system": system, "option": option}


def _quantize(name, batch, tokens, kv_heads, groups, bits=1, dtype="bf16", values="channel"):
    """The quantiser over one key or value tensor; `groups` > 0: the strided block of a fused projection output
    with that many query heads per kv head, 0: a contiguous tensor."""
    return {"name": name, "kind": "quantize", "batch": batch, "tokens": tokens, "kv_heads": kv_heads, "groups": groups,
            "bits": bits, "dtype": dtype, "values": values}


def _layer(name, batch, tiles, steps, system, text, bits=1, dtype="bf16"):
    """One attention layer of the 8B-shaped language model through the patched forward: prefill, then decode steps."""
    return {"name": name, "kind": "layer", "batch": batch, "tiles": tiles, "steps": steps, "system": system, "text": text,
            "bits": bits, "dtype": dtype}


def listed():
    return [
        # one sample, 1 024 cached tokens, fp16, no window yet: the smallest call, a single chat user
        _decode("decode-b1-kv1024-fp16", 1, 32, 8, 1024, 0, dtype="fp16"),
        # a small left-padded batch: additive mask, system prompt rows in the window, ragged lengths
        _decode("decode-b6-kv1789-masked", 6, 32, 8, 1789, 75, dtype="fp16", system=41, option="mask"),
        # the 8B-shaped layer at serving batch, 13 tiles and a 128-row window: the benchmark's own call, ...
        _decode("decode-b64-kv3328", 64, 32, 8, 3328, 128),
        # ... the same with two-bit codes, ...
        _decode("decode-b64-kv3328-2bit", 64, 32, 8, 3328, 128, bits=2),
        # ... and with values quantised per token
        _decode("decode-b64-kv3328-token-values", 64, 32, 8, 3328, 128, values="token"),
        # the 26B-shaped layer (six query heads per kv head), multi-image prompt, the step of a recorded graph
        _decode("decode-b16-kv9984-g6", 16, 48, 8, 9984, 105, system=41, option="device-rows"),
        # long context: the token axis is shared by several workgroups
        _decode("decode-b8-kv32768", 8, 32, 8, 32768, 0),
        # throughput serving, more work than fits the device at once
        _decode("decode-b256-kv3328", 256, 32, 8, 3328, 0),
        # prefill of one key tensor, read in place from the fused projection output
        _quantize("quantize-b64-t3328", 64, 3328, 8, 4),
        # a single long document
        _quantize("quantize-b1-t32768", 1, 32768, 8, 0),
        # prefill of one value tensor in the per-token layout
        _quantize("quantize-token-b64-t3328", 64, 3328, 8, 4, values="token"),
        # one layer through the patched forward, one tile per sample: prefill and sixteen tokens
        _layer("layer-b4-tile1-16-steps", 4, 1, 16, 41, 23),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("decode", "quantize", "layer"), (8, 4, 1))[0]
    bits = rng.choice((1, 1, 2))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind == "layer":
        c = _layer("", _log(rng, 1, 6), 1, rng.randint(4, 16), rng.randint(1, 41), rng.randint(1, 23), bits, dtype)
    elif kind == "quantize":
        heads = rng.choice((2, 4, 8))
        tokens = _log(rng, 64, 32768)
        batch = _log(rng, 1, max(1, min(64, 64 * 3328 * 8 // (tokens * heads))))
        c = _quantize("", batch, tokens, heads, rng.choice((0, 1, 2, 4, 6)), bits, dtype, rng.choice(("channel", "channel", "token")))
    else:
        heads = rng.choice((2, 4, 8))
        group = rng.choice((1, 2, 3, 4, 4, 6, 7, 8))
        tokens = _log(rng, 64, 32768)
        # at most the wide-batch case's tokens, in units of at most four query heads
        room = 128 * 3328 * 8 // (tokens * heads * bits * -(-group // 4))
        batch = _log(rng, 1, max(1, min(256, room)))
        rows = rng.choice((0, rng.randint(1, 128), rng.randint(129, 300)))
        option = rng.choice(("none", "none", "mask", "device-rows")) if rows else "none"
        c = _decode("", batch, heads * group, heads, tokens, rows, bits, dtype, rng.choice(("channel", "channel", "channel", "token")),
                    min(rows, 41) if rng.random() < 0.5 else 0, option)
    del c["name"]
    return c


def _keys(shape, g, dtype):
    """N(0, 1) keys (B, T, H, D) with four outlier channels per head, scaled by one to about ten."""
    k = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    heads = shape[2]
    gain = torch.ones((heads, D), device="cuda")
    for h in range(heads):
        ch = torch.randperm(D, generator=g, device="cuda")[:4]
        gain[h, ch] = 1.0 + 9.0 * torch.rand(4, generator=g, device="cuda") ** 2
    return k.mul_(gain.to(dtype))


def _prepare_decode(c, g):
    B, Hq, Hkv, T, R, bits, dt = c["batch"], c["q_heads"], c["kv_heads"], c["tokens"], c["rows"], c["bits"], DTYPES[c["dtype"]]
    ck, sk, zk = ops.quantize_pack(_keys((B, T, Hkv, D), g, dt), bits, CLIP_K[bits])
    v = torch.randn((B, T, Hkv, D), generator=g, device="cuda", dtype=dt)
    cv, sv, zv = ops.quantize_pack_token(v, bits) if c["values"] == "token" else ops.quantize_pack(v, bits, CLIP_V[bits])
    del v
    q = torch.randn((B, Hq, D), generator=g, device="cuda", dtype=dt)
    kr = vr = mask = r_dev = None
    if R:
        # the window is a view of a buffer with room for the tokens to come
        cap = R + max(256, R // 8)
        kr = torch.randn((B, Hkv, cap, D), generator=g, device="cuda", dtype=dt)
        vr = torch.randn((B, Hkv, cap, D), generator=g, device="cuda", dtype=dt)
        if c["option"] == "device-rows":
            r_dev = torch.full((1,), R, dtype=torch.int32, device="cuda")
        else:
            kr, vr = kr[:, :, :R], vr[:, :, :R]
    if c["option"] == "mask":
        pad = torch.randint(0, max(1, c["system"] // 2 + 1), (B, 1), generator=g, device="cuda")
        mask = torch.where(torch.arange(T + R, device="cuda") < pad, -1e4, 0.0)
    call = ops.DecodeCall(q, ck, cv, sk, zk, sv, zv, kr, vr, sprompt_len=c["system"], bits=bits, mask=mask, r_dev=r_dev,
                          v_mode=c["values"])
    return {"kind": "decode", "call": call}


def _prepare_quantize(c, g):
    B, T, H, dt = c["batch"], c["tokens"], c["kv_heads"], DTYPES[c["dtype"]]
    if c["groups"]:
        proj = torch.randn((B, T, H, c["groups"] + 2, D), generator=g, device="cuda", dtype=dt)
        x = proj[..., -1 if c["values"] == "token" else -2, :]
    else:
        x = _keys((B, T, H, D), g, dt)
    return {"kind": "quantize", "x": x, "bits": c["bits"], "token": c["values"] == "token"}


def _prepare_layer(c, g):
    cfg = InternLM2Config.internvl2_5_8b()
    dt = DTYPES[c["dtype"]]
    B, N = c["batch"], c["system"] + 256 * c["tiles"] + c["text"]
    with torch.device("cuda"):
        att = InternLM2Attention(cfg).to(dt).eval()
    for w in (att.wqkv.weight, att.wo.weight):
        w.data.normal_(0.0, cfg.hidden_size ** -0.5, generator=g)
    att.cq_image_token_num, att.cq_sprompt_len, att.cq_bits = 256 * c["tiles"], c["system"], c["bits"]
    x = torch.randn((B, N + c["steps"], cfg.hidden_size), generator=g, device="cuda", dtype=dt)
    pos = torch.arange(N + c["steps"], device="cuda")[None].repeat(B, 1)
    return {"kind": "layer", "att": att, "x": x, "pos": pos, "prompt": N}


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {"decode": _prepare_decode, "quantize": _prepare_quantize, "layer": _prepare_layer}[case["kind"]](case, g)


@torch.no_grad()
def run(state):
    if state["kind"] == "decode":
        return state["call"].run()
    if state["kind"] == "quantize":
        if state["token"]:
            return ops.quantize_pack_token(state["x"], state["bits"])
        return ops.quantize_pack(state["x"], state["bits"], CLIP_K[state["bits"]])
    forward, att, x, pos, n = ATTN_FORWARD_FUNCTIONS["calibquant"], state["att"], state["x"], state["pos"], state["prompt"]
    out, _, past = forward(att, x[:, :n], position_ids=pos[:, :n], use_cache=True)
    outs = [out]
    for i in range(n, x.shape[1]):
        out, _, past = forward(att, x[:, i:i + 1], position_ids=pos[:, i:i + 1], past_key_value=past, use_cache=True)
        outs.append(out)
    return outs + [past[0], past[1], att.encoded_features_k, att.encoded_features_v]


def work(case):
    c = case
    if c["kind"] == "decode":
        B, Hq, Hkv, T, R, bits = c["batch"], c["q_heads"], c["kv_heads"], c["tokens"], c["rows"], c["bits"]
        codes = 2 * B * Hkv * T * D * bits // 8
        stats = 2 * B * Hkv * D * 2 + (2 * B * Hkv * T * (D // 32) * 2 if c["values"] == "token" else 2 * B * Hkv * D * 2)
        mask = B * (T + R) * 4 if c["option"] == "mask" else 0
        return {"bytes": codes + stats + 2 * B * Hkv * R * D * 2 + 2 * B * Hq * D * 2 + mask, "flops": 4 * B * Hq * (T + R) * D}
    if c["kind"] == "quantize":
        n = c["batch"] * c["tokens"] * c["kv_heads"] * D
        stats = 2 * n // 32 * 2 if c["values"] == "token" else 2 * c["batch"] * c["kv_heads"] * D * 2
        return {"bytes": 2 * n + n * c["bits"] // 8 + stats, "flops": 4 * n}
    # layer: projections and causal attention; weights, hidden states in and out, codes and window written once
    B, N, steps, hidden, wide = c["batch"], c["system"] + 256 * c["tiles"] + c["text"], c["steps"], 4096, 6144
    rows = B * (N + steps)
    flops = 2 * rows * hidden * (wide + hidden) + 4 * B * 32 * D * (N * N // 2 + steps * (N + steps // 2))
    kv = 2 * B * 8 * (256 * c["tiles"] * D * c["bits"] // 8 + (c["system"] + c["text"] + steps) * D * 2)
    return {"bytes": 2 * hidden * (wide + hidden) + 2 * 2 * rows * hidden + kv, "flops": flops}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # About four times the distance to the same attention in 64 bits: 1.8e-3 to 2.4e-3 measured in bf16 (1.7e-3 of
    # it the rounding of the result), 0.6e-3 to 1.7e-3 in fp16.  The layer rounds its output projection once more.
    if case["kind"] == "layer":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 4e-3}
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 4e-3}
