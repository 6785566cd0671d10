"""The work that a user has this package do, as cases that can be timed.

Two entry points carry nearly all of it: `LutLinear.forward`, the quantised linear layer in its four
storage formats, called with one row per sequence while tokens are generated and with every row of
the prompt before that; and `LutDecoder.forward_token`, the graph-captured decode step of a whole
network.  `lutgemm.lutgemm_compute`, the uniform-quantisation function of the extension module, is
called by users of plain LUT-GEMM checkpoints.

A case is a dict of plain values:
  kind "linear":  LutLinear(K, N, wbit=bits, alpha_format=format) on `rows` rows of `dtype`; `group` is
                  the group length along K for format "rowwise_fp16", `row_groups` the number of output
                  row groups for the block formats; `alpha` says what the scales look like: "pow2" (what
                  the quantiser emits), "apot3" (sums of three powers of two) or "any" (least squares).
  kind "uniform": lutgemm_compute, scales and q_bias per group of `group` inputs.
  kind "decoder": LutDecoder of the stated geometry at position `position` of its cache.
"""
import math

import torch

from shiftaddllm_amd import native, workload
from shiftaddllm_amd.decode import DecoderConfig, LutDecoder
from shiftaddllm_amd.lut_gemm.quant import LutLinear, encode_apot_int8

DEVICE = "cuda:0"
VOCAB = 32000


def _linear(name, K, N, rows, format, bits, group=0, row_groups=0, alpha="pow2", bias=False, dtype="fp16"):
    return {"name": name, "kind": "linear", "K": K, "N": N, "rows": rows, "format": format, "bits": bits, "group": group,
            "row_groups": row_groups, "alpha": alpha, "bias": bias, "dtype": dtype}


def _decoder(name, batch, position, max_positions, layers=32, hidden=4096, intermediate=11008, heads=32, kv_heads=32, bits=0):
    return {"name": name, "kind": "decoder", "batch": batch, "position": position, "max_positions": max_positions,
            "layers": layers, "hidden": hidden, "intermediate": intermediate, "heads": heads, "kv_heads": kv_heads, "bits": bits}


def listed():
    return [
        # the first MLP layer of OPT-125m in the default storage, one generated token: the smallest call
        _linear("opt125m fc1, 1 token", 768, 3072, 1, "apot_int8", 3, row_groups=8, bias=True),
        # the second one on a prompt of 128 tokens
        _linear("opt125m fc2, prompt 128", 3072, 768, 128, "apot_int8", 3, row_groups=8, bias=True),
        # an attention projection of Llama-2-7B, one generated token
        _linear("llama7b q, 1 token", 4096, 4096, 1, "rowwise_fp16", 3, group=128),
        # gate_proj of Llama-2-13B with one scale per block of 8 columns, one generated token
        _linear("llama13b gate, 1 token", 5120, 13824, 1, "block_fp16", 2, row_groups=8),
        # gate_proj of Llama-2-70B, one generated token: the longest sign stream
        _linear("llama70b gate, 1 token", 8192, 28672, 1, "rowwise_fp16", 4, group=128),
        # its down_proj with 32 sequences in flight
        _linear("llama70b down, 32 rows", 28672, 8192, 32, "rowwise_fp16", 4, group=128),
        # a small batch on a layer whose sizes fit no tile, scales from least squares, a bfloat16 network
        _linear("ragged, 7 rows", 2208, 2964, 7, "rowwise_fp16", 3, group=96, alpha="any", bias=True, dtype="bf16"),
        # down_proj of Llama-2-13B in the default storage on a prompt of 512 tokens
        _linear("llama13b down, prompt 512", 13824, 5120, 512, "apot_int8", 2, row_groups=8),
        # gate_proj of Llama-2-7B on a full sequence, as in a perplexity run
        _linear("llama7b gate, prompt 2048", 4096, 11008, 2048, "rowwise_fp16", 3, group=128),
        # a uniformly quantised layer, one generated token
        {"name": "uniform 4096, 1 token", "kind": "uniform", "K": 4096, "N": 4096, "rows": 1, "bits": 4, "group": 128},
        # a token of Llama-2-7B with mixed bit widths at the end of 128 prompt and 128 generated ones
        _decoder("llama7b decode, batch 1", 1, 255, 256),
        # the same for eight sequences with a longer context
        _decoder("llama7b decode, batch 8", 8, 700, 1024),
    ]


# ---- more cases of the same ranges ---------------------------------------------------------------
MOST_MACS = 13824 * 5120 * 512   # rows * N * K of a drawn case
MOST_WEIGHTS = 28672 * 8192


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(v, of, least):
    return max(least, v // of * of)


def _draw_sizes(rng):
    """(K, N, rows): layers of 256 to 28672 inputs and outputs, one row in half of the cases, half of the
    others at most 64; sizes in half of the cases multiples of 128 as published networks have them."""
    while True:
        unit = rng.choice((True, False))
        K = _multiple(_log(rng, 256, 28672), 128 if unit else 32, 256)
        N = _multiple(_log(rng, 256, 28672), 128 if unit else 4, 256)
        pick = rng.random()
        rows = 1 if pick < 0.5 else _log(rng, 2, 64) if pick < 0.75 else _log(rng, 65, 2048)
        if K * N <= MOST_WEIGHTS and rows * K * N <= MOST_MACS:
            return K, N, rows


def _draw_group(rng, K):
    """A group length along K: 128 where it divides, otherwise one of the multiples of 32 that do."""
    fits = [g for g in range(32, min(K, 512) + 1, 32) if K % g == 0]
    return 128 if K % 128 == 0 and rng.random() < 0.7 else rng.choice(fits)


def _draw_row_groups(rng, K, N):
    fits = [r for r in (1, 2, 4, 8, 16) if N % (4 * r) == 0 and K % r == 0]
    return 8 if 8 in fits and rng.random() < 0.7 else rng.choice(fits)


def draw(rng):
    pick = rng.random()
    if pick < 0.7:
        K, N, rows = _draw_sizes(rng)
        format = rng.choice(("rowwise_fp16", "rowwise_fp16", "apot_int8", "apot_int8", "block_fp16", "block_shift_u16"))
        case = _linear("", K, N, rows, format, rng.choice((2, 3, 3, 4)), bias=rng.random() < 0.5,
                       dtype=rng.choice(("fp16", "fp16", "bf16", "fp32")))
        if format == "rowwise_fp16":
            case.update(group=_draw_group(rng, K), alpha=rng.choice(("pow2", "pow2", "any")))
        else:
            case.update(row_groups=_draw_row_groups(rng, K, N))
            case.update(alpha="apot3" if format == "block_shift_u16" else rng.choice(("pow2", "pow2", "apot3")))
    elif pick < 0.8:
        K, N, rows = _draw_sizes(rng)
        case = {"kind": "uniform", "K": K, "N": N, "rows": rows, "bits": rng.choice((2, 3, 4)), "group": _draw_group(rng, K)}
    else:
        heads = rng.choice((8, 16, 32, 40))
        hidden = 128 * heads
        max_positions = rng.choice((256, 512, 1024, 2048))
        batch = _log(rng, 1, 16)
        case = _decoder("", batch, rng.randrange(16, max_positions), max_positions, layers=rng.randint(2, 8), hidden=hidden,
                        intermediate=_multiple(int(hidden * rng.uniform(2.5, 3.6)), 128, 128), heads=heads,
                        kv_heads=rng.choice((heads, heads // 4 if heads % 4 == 0 else heads)), bits=rng.choice((0, 0, 2, 3, 4)))
    case.pop("name", None)
    return case


# ---- inputs --------------------------------------------------------------------------------------
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _signs(g, K, N, bits):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, bits, N), generator=g, device=DEVICE, dtype=torch.int32)


def _scales(g, kind, outer, bits, inner):
    """Scales [outer, bits, inner] as binary coding of N(0, 0.02) weights gives them: a base per group, about
    halving from plane to plane."""
    e = torch.randint(-8, -5, (outer, 1, inner), generator=g, device=DEVICE).float()
    a = torch.exp2(e - torch.arange(bits, device=DEVICE).float().view(1, bits, 1))
    if kind == "pow2":
        return a
    f = torch.rand((outer, bits, inner), generator=g, device=DEVICE)
    return a * (1.0 + f) if kind == "any" else a * (1.0 + torch.exp2(-1.0 - (f * 4).floor()) + 0.0625)


def _prepare_linear(case, g):
    K, N, bits = case["K"], case["N"], case["bits"]
    format = case["format"]
    group = case["group"] if format == "rowwise_fp16" else K // case["row_groups"]
    bias = (torch.randn(N, generator=g, device=DEVICE) * 0.1).half() if case["bias"] else None
    lin = LutLinear(K, N, group_size=group, wbit=bits, bias=bias, alpha_format=format).to(DEVICE)
    lin.binaryWeight.data = _signs(g, K, N, bits)
    if format == "rowwise_fp16":
        lin.alpha.data = _scales(g, case["alpha"], K // group, bits, N).half()
    elif format == "block_shift_u16":      # three shift fields of 0..7 each: sums of powers of two from 3 to 384
        s = torch.randint(0, 8, (3, K // 8, bits, case["row_groups"]), generator=g, device=DEVICE)
        lin.alpha.data = (s[0] | (s[1] << 3) | (s[2] << 6)).to(torch.int16)
    else:
        a = _scales(g, case["alpha"], K // 8, bits, case["row_groups"])
        lin.alpha.data = a.half() if format == "block_fp16" else encode_apot_int8(a)
    x = torch.randn((case["rows"], K), generator=g, device=DEVICE)
    if format == "block_shift_u16":        # (whole-number scales leave the range of fp16 results to the activations)
        x = x / 256
    return {"kind": "linear", "layer": lin.eval(), "x": x.to(_DTYPES[case["dtype"]])}


def _prepare_uniform(case, g):
    K, N, bits, groups = case["K"], case["N"], case["bits"], case["K"] // case["group"]
    alpha = (0.02 * (0.5 + torch.rand((groups, N), generator=g, device=DEVICE))).half()
    q_bias = (0.005 * torch.randn((groups, N), generator=g, device=DEVICE)).half()
    x = torch.randn((case["rows"], K), generator=g, device=DEVICE).half()
    return {"kind": "uniform", "signs": _signs(g, K, N, bits), "alpha": alpha, "q_bias": q_bias, "x": x, "N": N, "K": K,
            "bits": bits, "groups": groups}


def _quant_config(case):
    return workload.mixed_bit_config(case["layers"]) if case["bits"] == 0 else None


def _prepare_decoder(case, g, seed):
    cfg = DecoderConfig(vocab_size=VOCAB, hidden=case["hidden"], intermediate=case["intermediate"], layers=case["layers"],
                        heads=case["heads"], kv_heads=case["kv_heads"], max_positions=case["max_positions"])
    model = LutDecoder(cfg, _quant_config(case), batch=case["batch"], seed=seed, device=DEVICE, default_bits=case["bits"] or 3)
    model.k_cache.normal_(generator=g)     # what the tokens before this one left
    model.v_cache.normal_(generator=g)
    model.capture()
    ids = torch.randint(0, VOCAB, (case["batch"],), generator=g, device=DEVICE)
    return {"kind": "decoder", "model": model, "ids": ids, "position": case["position"]}


def prepare(case, seed):
    g = _generator(seed)
    if case["kind"] == "linear":
        return _prepare_linear(case, g)
    if case["kind"] == "uniform":
        return _prepare_uniform(case, g)
    return _prepare_decoder(case, g, seed)


def run(state):
    if state["kind"] == "linear":
        with torch.no_grad():
            return state["layer"](state["x"])
    if state["kind"] == "uniform":
        out = torch.zeros((state["x"].shape[0], state["N"]), dtype=torch.float16, device=DEVICE)
        native.lutgemm.lutgemm_compute(out, state["signs"], state["alpha"], state["q_bias"], state["x"], state["N"], state["K"],
                                       state["bits"], state["groups"])
        return out
    model = state["model"]
    logits = model.forward_token(state["ids"], state["position"])
    return {"logits": logits, "k_cache": model.k_cache, "v_cache": model.v_cache}


# ---- what a pass cannot do without ---------------------------------------------------------------
def _layer_bytes(K, N, bits, scale_bytes, rows, in_bytes, out_bytes):
    return K * N * bits // 8 + scale_bytes + rows * (K * in_bytes + N * out_bytes)


def work(case):
    if case["kind"] == "decoder":
        h, i, B = case["hidden"], case["intermediate"], case["batch"]
        kv = case["kv_heads"] * (h // case["heads"])
        shapes = {"self_attn.q_proj": (h, h), "self_attn.k_proj": (h, kv), "self_attn.v_proj": (h, kv), "self_attn.o_proj": (h, h),
                  "mlp.gate_proj": (h, i), "mlp.up_proj": (h, i), "mlp.down_proj": (i, h)}
        config = _quant_config(case)
        total = flops = 0
        for layer in range(case["layers"]):
            for name, (K, N) in shapes.items():
                bits = config[f"model.layers.{layer}.{name}"]["bits"] if config else case["bits"]
                total += K * N * bits // 8 + K // 128 * bits * N * 2
                flops += 2 * B * K * N
            total += 2 * B * (case["position"] + 2) * kv * 2     # keys and values read, the new ones written
            flops += 4 * B * (case["position"] + 1) * h
        total += 2 * (VOCAB * h + B * h + B * VOCAB)             # output matrix, embedding rows, logits
        return {"bytes": total, "flops": flops + 2 * B * VOCAB * h}
    K, N, bits, rows = case["K"], case["N"], case["bits"], case["rows"]
    if case["kind"] == "uniform":
        scales, io = 2 * 2 * (K // case["group"]) * N, 2
    elif case["format"] == "rowwise_fp16":
        scales, io = 2 * (K // case["group"]) * bits * N, 4 if case["dtype"] == "fp32" else 2
    else:
        scales = (3 if case["format"] == "apot_int8" else 2) * (K // 8) * bits * case["row_groups"]
        io = 4 if case["dtype"] == "fp32" else 2
    bias = 2 * N if case.get("bias") else 0
    return {"bytes": _layer_bytes(K, N, bits, scales + bias, rows, io, io), "flops": 2 * rows * K * N}


def tolerance(case):
    if case["kind"] == "decoder":
        # fp16 activations through every block: one rounding more or less is amplified from block to block
        return {"rel": 1.5e-2, "max": 0.1}
    if case.get("dtype") == "bf16":
        return {"rel": 5e-3, "max": 2e-2}     # results rounded to bfloat16
    return {"rel": 1e-3, "max": 6e-3}         # sums of 32 bits, results rounded to fp16
