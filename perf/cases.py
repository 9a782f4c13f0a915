"""The calls whose speed matters to a user of this package, with their inputs and how exact their results are.

Three kinds of work, each through the public entry points: static W8A8 linears on bytes (`QLinear`, alone and
between the Quantize/DequantizeLinear nodes of an exported graph), weight-only-packed linears on f32 rows
(`PackedLinear` under DYNAMIC_I8, eight- and four-bit weights), and the decoder built from them
(`W8A8Decoder`: prompts and token steps).

A case's fields:
  kind     "qlinear" | "linear" | "prompt" | "steps"
  rows, k, n                     extents of a linear (decoder: rows = sequences served together)
  form     qlinear: "bytes" (int8 in, int8 out), "rows" (one input scale per row, f32 bias, int8 out),
           "f32" (QuantizeLinear -> QLinear -> DequantizeLinear on f32 rows)
  unsigned, zero_points          qlinear: U8 activations; weights with zero points
  bits, group, grouped           linear: weight width, scale group, scales that differ from group to group
  layers, small, tokens, steps   decoder: depth, the narrow widths, prompt length, steps behind the prompt
"""
from __future__ import annotations

import numpy as np
import torch

import volvoxai_amd as vx
from volvoxai_amd.decoder import DecoderConfig, W8A8Decoder, pack_w4_words, pack_w8_words


def listed():
    return [
        # one row of a small static layer: nothing but latency (a keyword spotter, a classifier head)
        dict(name="qlinear_row", kind="qlinear", form="bytes", rows=1, k=1024, n=1024, unsigned=False, zero_points=False),
        # an exported graph's sandwich on a small batch of odd extents, unsigned activations, zero points
        dict(name="qlinear_ragged_f32", kind="qlinear", form="f32", rows=77, k=1001, n=1531, unsigned=True,
             zero_points=True),
        # prompts through a static layer: per-token scales, requantized; a short one and the largest
        dict(name="qlinear_prompt_512", kind="qlinear", form="rows", rows=512, k=4096, n=4096, unsigned=False,
             zero_points=False),
        dict(name="qlinear_prompt_4096", kind="qlinear", form="rows", rows=4096, k=4096, n=4096, unsigned=False,
             zero_points=False),
        # a feed-forward projection in decode: one stream, and a batch of streams
        dict(name="linear_row", kind="linear", rows=1, k=4096, n=14336, bits=8, group=128, grouped=True),
        dict(name="linear_batch_24", kind="linear", rows=24, k=4096, n=14336, bits=8, group=128, grouped=True),
        # the same with four-bit weights and a few streams
        dict(name="linear_w4_rows_4", kind="linear", rows=4, k=4096, n=14336, bits=4, group=128, grouped=True),
        # a long prompt through a down projection, eight-bit weights quantized per channel
        dict(name="linear_prompt_2048", kind="linear", rows=2048, k=14336, n=4096, bits=8, group=128, grouped=False),
        # a prompt of odd length, four-bit weights in fine groups, extents that fit no tile
        dict(name="linear_w4_prompt_333", kind="linear", rows=333, k=3000, n=5001, bits=4, group=32, grouped=True),
        # the decoder: 32 prompts at once; a batch served for 32 steps behind its prompts; a single stream
        dict(name="decoder_prompt_32x128", kind="prompt", rows=32, layers=28, small=False, tokens=128, steps=0),
        dict(name="decoder_steps_32", kind="steps", rows=32, layers=28, small=False, tokens=128, steps=32),
        dict(name="decoder_steps_1", kind="steps", rows=1, layers=28, small=False, tokens=128, steps=32),
    ]


def _log_int(rng, low, high, multiple=1):
    v = int(round(low * (high / low) ** rng.random()))
    return max(low, min(high, max(1, round(v / multiple)) * multiple))


def draw(rng):
    kind = rng.choice(["qlinear", "qlinear", "linear", "linear", "linear", "prompt", "steps"])
    if kind == "qlinear":
        step = rng.choice([1, 16, 256])
        form = rng.choice(["bytes", "rows", "f32"])
        return dict(kind=kind, form=form, rows=_log_int(rng, 1, 4096), k=_log_int(rng, 256, 4096, step),
                    n=_log_int(rng, 256, 4096, step), unsigned=form != "rows" and rng.random() < 0.5,
                    zero_points=form != "rows" and rng.random() < 0.3)
    if kind == "linear":
        step = rng.choice([1, 32, 512])
        return dict(kind=kind, rows=_log_int(rng, 1, 2048), k=_log_int(rng, 512, 14336, step),
                    n=_log_int(rng, 256, 14336 if rng.random() < 0.5 else 4096, step), bits=rng.choice([8, 8, 4]),
                    group=rng.choice([32, 64, 128, 128, 256]), grouped=rng.random() < 0.7)
    small = rng.random() < 0.3
    return dict(kind=kind, rows=_log_int(rng, 1, 32), layers=rng.randint(2, 8), small=small,
                tokens=rng.randint(9, 190), steps=0 if kind == "prompt" else rng.randint(8, 40))


# ---- inputs -----------------------------------------------------------------------------------------

def _normal(gen, shape, std=1.0):
    return torch.randn(shape, generator=gen, device="cuda") * std


def _uniform(gen, shape, low, high):
    return torch.rand(shape, generator=gen, device="cuda") * (high - low) + low


def _weights(gen, n, k, bits):
    """Round-to-nearest codes of normally distributed weights, the largest of a few thousand at full scale."""
    top = 2 ** (bits - 1) - 1
    return (_normal(gen, (n, k), top / 3.5)).round_().clamp_(-top, top).to(torch.int8).cpu().numpy()


def _group_scales(gen, n, k, group, grouped):
    groups = (k + group - 1) // group
    scales = _uniform(gen, (n, 1), 0.002, 0.01).expand(n, groups)
    if grouped:
        scales = scales * _uniform(gen, (n, groups), 0.7, 1.0)
    return scales.contiguous().cpu().numpy()


def _activations(gen, rows, k):
    """f32 rows with a few strong channels, as the inputs of a transformer's projections have them."""
    x = _normal(gen, (rows, k))
    x[:, torch.randperm(k, generator=gen, device="cuda")[:max(1, k // 100)]] *= 20.0
    return x


def _config(case):
    if case["small"]:
        return DecoderConfig(layers=case["layers"], hidden=512, q_heads=8, kv_heads=4, head_dim=64, inter=1536,
                             vocab=8000)
    return DecoderConfig(layers=case["layers"])


def _decoder_weights(gen, cfg):
    """Random weights of the architecture in the form W8A8Decoder takes (volvoxai_amd.decoder.init_weights)."""
    def linear(n, k, gain=1.0):
        # (scales that keep a row of unit variance near unit variance, as trained weights do)
        scales = _group_scales(gen, n, k, cfg.group, False) * np.float32(4.6 * gain / np.sqrt(k))
        return {"w": _weights(gen, n, k, 8), "scales": scales}

    # a layer of a trained model adds a few percent to its residual stream, the less the deeper the model is
    branch = 0.4 / np.sqrt(2.0 * cfg.layers)

    def gain():
        return _uniform(gen, (cfg.hidden,), 0.5, 1.5).cpu().numpy()

    layers = [{"norm1": gain(), "qkv": linear(cfg.q_dim + 2 * cfg.kv_dim, cfg.hidden),
               "o": linear(cfg.hidden, cfg.q_dim, branch), "norm2": gain(), "gate_up": linear(2 * cfg.inter, cfg.hidden),
               "down": linear(cfg.hidden, cfg.inter, branch)} for _ in range(cfg.layers)]
    return {"embedding": _normal(gen, (cfg.vocab, cfg.hidden)).cpu().numpy(), "layers": layers, "norm_f": gain(),
            "lm_head": linear(cfg.vocab, cfg.hidden)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = dict(case)
    if case["kind"] == "qlinear":
        rows, k, n = case["rows"], case["k"], case["n"]
        w = _weights(gen, n, k, 8)
        zps = np.zeros(n, np.int32)
        if case["zero_points"]:
            zps = torch.randint(-9, 10, (n,), generator=gen, device="cuda").to(torch.int32).cpu().numpy()
        scales = _uniform(gen, (n,), 0.005, 0.02).cpu().numpy()
        bias = torch.randint(-2000, 2001, (n,), generator=gen, device="cuda").to(torch.int32).cpu().numpy()
        s["linear"] = vx.QLinear(w, scales, zps, None if case["form"] == "rows" else bias, vx.DTYPE_I8)
        s["zp_in"] = 121 if case["unsigned"] else 0
        s["in_dtype"] = vx.DTYPE_U8 if case["unsigned"] else vx.DTYPE_I8
        # activations of standard deviation 30 codes; the output scale puts one of the output at about 40
        s["s_in"], s["s_out"] = 0.02, float(0.02 * 0.0125 * 30 * 36 * np.sqrt(k) / 40)
        if case["form"] == "f32":
            s["x"] = _normal(gen, (rows, k), 30 * s["s_in"])
        else:
            low, high, kind = (0, 255, torch.uint8) if case["unsigned"] else (-127, 127, torch.int8)
            s["x"] = (_normal(gen, (rows, k), 30.0) + s["zp_in"]).round_().clamp_(low, high).to(kind)
        if case["form"] == "rows":
            s["row_scales"] = _uniform(gen, (rows,), 0.01, 0.03)
            s["bias_f32"] = _normal(gen, (n,), s["s_out"])
        s["ctx"] = vx.Context(0, torch.cuda.current_stream())
    elif case["kind"] == "linear":
        rows, k, n, bits = case["rows"], case["k"], case["n"], case["bits"]
        words = (pack_w8_words if bits == 8 else pack_w4_words)(_weights(gen, n, k, bits))
        scales = _group_scales(gen, n, k, case["group"], case["grouped"])
        bias = _normal(gen, (n,), 0.1).cpu().numpy()
        s["linear"] = vx.PackedLinear(words, scales, bias, k, n, case["group"], weight_bits=bits)
        s["x"] = _activations(gen, rows, k)
        s["ctx"] = vx.Context(0, torch.cuda.current_stream())
    else:
        cfg = _config(case)
        s["decoder"] = dec = W8A8Decoder(cfg, _decoder_weights(gen, cfg), case["rows"])
        s["prompt"] = torch.randint(0, cfg.vocab, (case["rows"], case["tokens"]), generator=gen, device="cuda")
        if case["kind"] == "steps":
            s["ids"] = torch.randint(0, cfg.vocab, (case["steps"], case["rows"]), generator=gen,
                                     device="cuda").to(torch.int32)
            dec.capture()
            s["step_logits"] = dec.last_logits  # a captured step writes its logits here
            s["logits"] = torch.empty((case["steps"], case["rows"], cfg.vocab), device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    if s["kind"] == "qlinear":
        lin, ctx, x = s["linear"], s["ctx"], s["x"]
        if s["form"] == "rows":
            ok, y = lin.forward_rowscale(ctx, x, s["row_scales"], s["s_out"], 0, bias_f32=s["bias_f32"])
        elif s["form"] == "f32":
            ok, y, _ = lin.forward_f32(ctx, x, s["s_in"], s["zp_in"], s["s_out"], 0, input_dtype=s["in_dtype"])
        else:
            ok, y = lin.forward(ctx, x, s["s_in"], s["zp_in"], s["s_out"], 0, input_dtype=s["in_dtype"])
        if ok != 1:
            raise RuntimeError("the linear declined the call")
        return y
    if s["kind"] == "linear":
        status, y = s["linear"].forward_f32(s["ctx"], s["x"])
        if status != 0:
            raise RuntimeError("the linear declined the call")
        return y
    dec = s["decoder"]
    dec.prefill(s["prompt"])
    if s["kind"] == "prompt":
        return {"logits": dec.last_logits, "k_cache": dec.k_cache, "v_cache": dec.v_cache}
    # a program that chooses the ids itself (sampling, or scoring a given text), one step at a time
    with torch.cuda.stream(dec.stream):
        for ids, logits in zip(s["ids"], s["logits"]):
            dec.tokens.copy_(ids)
            dec.decode(1)
            logits.copy_(s["step_logits"])
    return {"logits": s["logits"], "k_cache": dec.k_cache, "v_cache": dec.v_cache}


def work(case):
    if case["kind"] in ("qlinear", "linear"):
        rows, k, n = case["rows"], case["k"], case["n"]
        flops = 2.0 * rows * k * n
        if case["kind"] == "linear":
            groups = (k + case["group"] - 1) // case["group"] if case["grouped"] else 1
            return {"bytes": n * k * case["bits"] / 8 + 4.0 * n * (groups + 1) + 4.0 * rows * (k + n), "flops": flops}
        wide = 4 if case["form"] == "f32" else 1
        return {"bytes": n * k + 12.0 * n + wide * rows * (k + n), "flops": flops}
    cfg = _config(case)
    rows, tokens, steps = case["rows"], case["tokens"], case["steps"]
    layer = cfg.hidden * (cfg.q_dim + 2 * cfg.kv_dim) + cfg.q_dim * cfg.hidden + 3 * cfg.hidden * cfg.inter
    weights = cfg.layers * layer + cfg.vocab * cfg.hidden
    slot = 2 * 4 * cfg.kv_dim * cfg.layers * rows  # key and value bytes of one position, all layers
    seen = sum(tokens + i + 1 for i in range(steps))
    attended = tokens * (tokens + 1) / 2 + seen
    return {"bytes": (1 + steps) * weights + slot * (tokens + seen) + 4.0 * rows * cfg.vocab * (1 + steps),
            "flops": 2.0 * rows * ((tokens + steps) * cfg.layers * layer + (1 + steps) * cfg.vocab * cfg.hidden)
            + 4.0 * rows * cfg.layers * cfg.q_dim * attended}


def tolerance(case):
    # A linear's sums are exact integers and its few f32 roundings come in a fixed order: the same bits.
    if case["kind"] in ("qlinear", "linear"):
        return "exact"
    # A decoder's attention sums in f32 in an order of its own, and a value next to a rounding boundary of the
    # int8 preparation behind it then takes the neighbouring code.  Measured by moving every embedding to the
    # next f32: 2-norm 0.010-0.013 of the logits' and 0.003-0.009 of the caches', largest difference 0.14.
    return {"rel": 0.03, "max": 0.5}
