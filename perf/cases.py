"""Performance cases of the quantized-linear framework: what a program that
serves or prepares an int4 / int8 model has it do, through ``metal_native``'s
public entry points.

Kinds of case (``case["kind"]``):

* ``linear`` -- one ``dequant_matmul`` over ``m`` rows, from a single decode
  row to a 4096-token prefill chunk, with the epilogue of its layer;
* ``vecmat`` -- ``matmul`` of a few rows with un-quantized weights (the
  layers a checkpoint leaves in fp16 or fp32);
* ``weights`` -- quantize one fp16 weight at load time and make the fp16 copy
  that ``QuantizedLinear.dequantized_weight`` hands out;
* ``decode_step`` -- one token through a whole synthetic decoder, replayed
  from the HIP graph that a decode loop keeps.

Inputs are random, made on the GPU from the seed alone: activations N(0, 1)
(what an RMSNorm leaves), int4 nibbles U{0..15} with scales U(0.005, 0.02) and
integer zero-points, int8 weights U{-127..127} with scales U(0.001, 0.01) and
zeros of 0.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "metal-native_amd"))

import metal_native as mn  # noqa: E402
from metal_native.decoder import DecoderConfig, SyntheticDecoder  # noqa: E402

DEVICE = "cuda:0"


def _linear(name, m, k, n, g, quant="int4", epilogue="none"):
    c = {"kind": "linear", "m": m, "k": k, "n": n, "g": g, "quant": quant, "epilogue": epilogue}
    return {"name": name, **c} if name else c


def listed():
    return [
        # batch-1 decode of a small model (Qwen2.5-0.5B gate projection): latency and the call itself
        _linear("decode_gate_0p5b_m1", 1, 896, 4864, 64),
        # batch-1 decode of a 7B model's longest rows (Qwen2.5-7B down projection)
        _linear("decode_down_7b_m1", 1, 18944, 3584, 128),
        # a decode batch whose size is what the scheduler happened to have (7B fused QKV with its bias)
        _linear("decode_qkv_7b_m13", 13, 3584, 4608, 128, epilogue="bias"),
        # a wide decode batch through per-channel int8 gate/up with SwiGLU: the heaviest weight read of one call
        _linear("decode_gateup_7b_int8_m64", 64, 3584, 37888, 3584, "int8", "swiglu"),
        # a few speculative tokens for each of several sequences (7B down projection onto the residual stream)
        _linear("verify_down_7b_m37", 37, 18944, 3584, 128, epilogue="residual"),
        # an ordinary prompt (Llama-3.2-3B fused QKV at 512 tokens)
        _linear("prefill_qkv_3b_m512", 512, 3072, 5120, 128),
        # a prompt of ragged length into few columns, finer groups of int8 (0.5B down projection)
        _linear("prefill_down_0p5b_int8_m301", 301, 4864, 896, 64, "int8"),
        # a prompt of ragged length over the longest rows (7B down projection onto the residual stream)
        _linear("prefill_down_7b_m777", 777, 18944, 3584, 128, epilogue="residual"),
        # a full prefill chunk through the widest layer (7B gate/up with SwiGLU): the largest call
        _linear("prefill_gateup_7b_m4096", 4096, 3584, 37888, 128, epilogue="swiglu"),
        # a layer left in fp16, decoding one row
        {"name": "vecmat_fp16_m1", "kind": "vecmat", "m": 1, "k": 3584, "n": 18944, "dtype": "float16", "layout": "nk"},
        # quantizing one layer while a checkpoint loads, and its fp16 copy (7B down projection)
        {"name": "weights_int4_7b_down", "kind": "weights", "k": 18944, "n": 3584, "g": 128, "quant": "int4"},
        # one token of a 7B model after a 512-token prompt
        {"name": "decode_step_7b_512", "kind": "decode_step", "layers": 28, "d": 3584, "heads": 28, "kv_heads": 4,
         "head_dim": 128, "ffn": 18944, "vocab": 152064, "g": 128, "context": 512, "max_len": 576},
    ]


# (K, N) of the projections of the models the listed cases come from; SwiGLU
# layers give gate and up rows together
_LAYERS = [(896, 1152), (896, 896), (896, 9728), (4864, 896), (3072, 5120), (3072, 3072), (3584, 4608), (3584, 3584),
           (3584, 37888), (18944, 3584)]
_MOST = 4096 * 3584 * 37888   # multiply-adds of the largest listed linear


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["linear", "vecmat", "weights", "decode_step"], [13, 3, 2, 2])[0]
    if kind == "vecmat":
        return {"kind": kind, "m": rng.randint(1, 8), "k": 8 * _log_int(rng, 64, 2368), "n": 8 * _log_int(rng, 64, 2368),
                "dtype": rng.choice(["float16", "float16", "float32"]), "layout": rng.choice(["nk", "nk", "kn"])}
    if kind == "weights":
        k, n = 128 * _log_int(rng, 7, 148), _log_int(rng, 512, 18944)
        return {"kind": kind, "k": k, "n": n, "g": rng.choice([32, 64, 128]), "quant": rng.choice(["int4", "int8"])}
    if kind == "decode_step":
        small = rng.random() < 0.4
        context = _log_int(rng, 16, 3900)
        c = {"kind": kind, "layers": rng.randint(2, 28), "context": context,
             "max_len": min(4096, context + rng.randint(1, 256))}
        if small:   # 0.5B shapes
            return {**c, "d": 896, "heads": 14, "kv_heads": 2, "head_dim": 64, "ffn": 4864, "vocab": 151936, "g": 64}
        return {**c, "d": 3584, "heads": 28, "kv_heads": 4, "head_dim": 128, "ffn": 18944, "vocab": 152064, "g": 128}
    m = _log_int(rng, 1, 4096)
    if rng.random() < 0.5:
        k, n = rng.choice(_LAYERS)
    else:       # other models and shards of these: K in whole 32s, any even N
        k, n = 32 * _log_int(rng, 16, 592), 2 * _log_int(rng, 256, 18944)
    while m * k * n > _MOST:
        n = max(512, n // 4 * 2)
        if n == 512:
            break
    quant = rng.choice(["int4", "int4", "int8"])
    groups = [g for g in (32, 64, 128) if k % g == 0] + ([k] if quant == "int8" else [])
    epilogue = rng.choice(["none", "none", "bias", "residual", "bias_silu", "swiglu"])
    return _linear(None, m, k, n, rng.choice(groups), quant, epilogue)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return gen


def _quantized(gen, k, n, g, quant):
    groups = -(-k // g)
    if quant == "int4":
        w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEVICE, generator=gen)
        s = (torch.rand((n, groups), device=DEVICE, generator=gen) * 0.015 + 0.005).half()
        zp = torch.randint(0, 16, (n, groups), device=DEVICE, generator=gen).float()
        z = ((zp - 8.0) * s.float()).half()
    else:
        w = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=DEVICE, generator=gen)
        s = (torch.rand((n, groups), device=DEVICE, generator=gen) * 0.009 + 0.001).half()
        z = torch.zeros_like(s)
    return w, s, z


def _linear_inputs(case, seed):
    gen = _generator(seed)
    m, k, n = case["m"], case["k"], case["n"]
    weights = _quantized(gen, k, n, case["g"], case["quant"])
    x = torch.randn((m, k), device=DEVICE, generator=gen).half()
    extra = {}
    if case["epilogue"].startswith("bias"):
        extra["bias"] = torch.randn(n, device=DEVICE, generator=gen).half()
    elif case["epilogue"] == "residual":
        extra["residual"] = torch.randn((m, n), device=DEVICE, generator=gen).half()
    return x, weights, extra


def _vecmat_inputs(case, seed):
    gen = _generator(seed)
    dtype = getattr(torch, case["dtype"])
    shape = (case["n"], case["k"]) if case["layout"] == "nk" else (case["k"], case["n"])
    a = torch.randn((case["m"], case["k"]), device=DEVICE, generator=gen).to(dtype)
    b = (torch.randn(shape, device=DEVICE, generator=gen) * 0.02).to(dtype)
    return a, b


def _float_weight(case, seed):
    return (torch.randn((case["n"], case["k"]), device=DEVICE, generator=_generator(seed)) * 0.05).half()


def _decoder(case, seed):
    cfg = DecoderConfig(layers=case["layers"], d=case["d"], heads=case["heads"], kv_heads=case["kv_heads"],
                        head_dim=case["head_dim"], ffn=case["ffn"], vocab=case["vocab"], group_size=case["g"],
                        max_len=case["max_len"])
    model = SyntheticDecoder(cfg, DEVICE, seed=seed, prefilled=case["context"])
    token = seed % case["vocab"]
    return model, token, case["context"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, (w, s, z), extra = _linear_inputs(case, seed)
        epilogue = None if case["epilogue"] == "none" else case["epilogue"]
        return {"kind": kind, "x": x, "w": w, "s": s, "z": z, "g": case["g"], "quant": case["quant"],
                "kw": {"epilogue": epilogue, **extra}}
    if kind == "vecmat":
        a, b = _vecmat_inputs(case, seed)
        return {"kind": kind, "a": a, "b": b, "nk": case["layout"] == "nk"}
    if kind == "weights":
        return {"kind": kind, "w": _float_weight(case, seed), "g": case["g"], "quant": case["quant"]}
    # one decode step at a fixed position, captured as a decode loop captures it
    model, token, context = _decoder(case, seed)
    tok = torch.tensor([token], dtype=torch.int64, device=DEVICE)
    pos = torch.tensor([context], dtype=torch.int64, device=DEVICE)
    model.start_chain(tok)
    stream = torch.cuda.Stream(DEVICE)
    stream.wait_stream(torch.cuda.current_stream(DEVICE))
    with torch.cuda.stream(stream):
        model.step(tok, pos, x_in=model.x0)
    torch.cuda.synchronize(DEVICE)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        logits = model.step(tok, pos, x_in=model.x0)
    return {"kind": kind, "graph": graph, "logits": logits, "kv": model.kv, "model": model, "tok": tok, "pos": pos}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "linear":
        return mn.dequant_matmul(state["x"], state["w"], state["s"], state["z"], state["g"], state["quant"], **state["kw"])
    if kind == "vecmat":
        return mn.matmul(state["a"], state["b"], False, state["nk"])
    if kind == "weights":
        packed, scales, zeros = mn.quantize(state["w"], state["g"], state["quant"])
        return packed, scales, zeros, mn.dequantize(packed, scales, zeros, state["g"], state["quant"])
    state["graph"].replay()
    return state["logits"], state["kv"]


def _weight_bytes(k, n, g, quant):
    groups = -(-k // g)
    # int8 zeros are part of the call's operands too
    return (n * k // 2 if quant == "int4" else n * k) + 4 * n * groups


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        out = n // 2 if case["epilogue"] == "swiglu" else n
        extra = 2 * n if case["epilogue"].startswith("bias") else 2 * m * n if case["epilogue"] == "residual" else 0
        return {"bytes": _weight_bytes(k, n, case["g"], case["quant"]) + 2 * m * k + 2 * m * out + extra,
                "flops": 2 * m * n * k}
    if kind == "vecmat":
        size = 2 if case["dtype"] == "float16" else 4
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": size * (n * k + m * k + m * n), "flops": 2 * m * n * k}
    if kind == "weights":
        # the fp16 weight read, the quantized one written and read, its fp16 copy written
        return {"bytes": 4 * case["n"] * case["k"] + 2 * _weight_bytes(case["k"], case["n"], case["g"], case["quant"]),
                "flops": 0}
    d, ffn, dh = case["d"], case["ffn"], case["head_dim"]
    nq, nkv = case["heads"] * dh, case["kv_heads"] * dh
    shapes = [(d, nq + 2 * nkv), (nq, d), (d, 2 * ffn), (ffn, d)]
    layer = sum(_weight_bytes(k, n, case["g"], "int4") for k, n in shapes)
    macs = case["layers"] * (sum(k * n for k, n in shapes) + 2 * nq * (case["context"] + 1)) + d * case["vocab"]
    kv = case["layers"] * 2 * nkv * 2 * (case["context"] + 1)
    return {"bytes": case["layers"] * layer + _weight_bytes(d, case["vocab"], case["g"], "int4") + kv + 2 * case["vocab"],
            "flops": 2 * macs}


def tolerance(case):
    """Each is about four times the distance measured between the path and
    ``exact``: one fp16 rounding of the result (2.1e-4 of it), with SwiGLU also
    those of gate and up (3.6e-4); fp32 sums in another order (1e-6)."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 1.5e-3} if case["epilogue"] == "swiglu" else {"rel": 1e-3}
    if kind == "vecmat":
        return {"rel": 1e-3} if case["dtype"] == "float16" else {"rel": 1e-5}
    if kind == "weights":
        return "exact"
    # fp16 roundings of every layer travel on through the layers that follow (1.2e-3 after 28)
    return {"rel": 5e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _dequantized(w, s, z, g, quant, k):
    """The fp16 weights that the storage format stands for: q * s rounded,
    minus z rounded (their exact values, as float64)."""
    if quant == "int4":
        q = torch.stack((w & 15, w >> 4), dim=-1).reshape(w.shape[0], k).to(torch.float16) - 8.0
    else:
        q = w.to(torch.float16)
    group = torch.arange(k, device=w.device) // g
    return (q * s[:, group] - z[:, group]).double()


def _product(x, w, s, z, g, quant):
    """x [m, k] float64 times the dequantized weights' transpose, by row blocks."""
    k = x.shape[1]
    rows = max(1, (1 << 28) // k)
    return torch.cat([x @ _dequantized(w[i:i + rows], s[i:i + rows], z[i:i + rows], g, quant, k).t().contiguous()
                      for i in range(0, w.shape[0], rows)], dim=1)


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _exact_linear(case, seed):
    x, (w, s, z), extra = _linear_inputs(case, seed)
    y = _product(x.double(), w, s, z, case["g"], case["quant"])
    if "bias" in extra:
        y = y + extra["bias"].double()
    if case["epilogue"] == "bias_silu":
        y = _silu(y)
    elif case["epilogue"] == "residual":
        y = y + extra["residual"].double()
    elif case["epilogue"] == "swiglu":
        half = case["n"] // 2
        y = _silu(y[:, :half]) * y[:, half:]
    return y


def _exact_weights(case, seed):
    """The quantizer's formulas are defined step by step in fp32 (fp16
    scales), and its bytes follow from them: the fp16 copy in 64 bits."""
    n, k, g = case["n"], case["k"], case["g"]
    w = _float_weight(case, seed).float().reshape(n, k // g, g)
    if case["quant"] == "int4":
        lo, hi = w.amin(-1), w.amax(-1)
        s = ((hi - lo) / 15.0).half()
        sf = s.float()
        zp = torch.round(-lo / sf).clamp(0, 15)
        q = (torch.round(w / sf[..., None]) + zp[..., None]).clamp(0, 15) - 8.0
        z = ((zp - 8.0) * s.float()).half()
    else:
        s = (w.abs().amax(-1) / 127.0).half()
        q = torch.round(w / s.float()[..., None]).clamp(-127, 127)
        z = torch.zeros_like(s)
    copy = (q.half() * s[..., None] - z[..., None]).reshape(n, k)
    return None, s.double(), z.double(), copy.double()


def _exact_decode_step(case, seed):
    model, token, pos = _decoder(case, seed)
    H, KVH, dh, eps = case["heads"], case["kv_heads"], case["head_dim"], model.cfg.eps
    f64 = torch.float64

    def lin(x, ql):
        y = _product(x, ql.wp, ql.scales, ql.zeros, ql.g, "int4")
        return y if ql.bias is None else y + ql.bias.double()

    def norm(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()

    def rope(v):
        half = dh // 2
        return v * cos + torch.cat([-v[:, half:], v[:, :half]], dim=-1) * sin

    cos, sin = model.cos[pos].double(), model.sin[pos].double()
    x = model.embed[token:token + 1].double()
    kv = model.kv.to(f64)
    for li, layer in enumerate(model.layers):
        qkv = lin(norm(x, layer["ln1"]), layer["qkv"])[0]
        q = rope(qkv[:H * dh].view(H, dh))
        kv[li, 0, :, pos] = rope(qkv[H * dh:(H + KVH) * dh].view(KVH, dh))
        kv[li, 1, :, pos] = qkv[(H + KVH) * dh:].view(KVH, dh)
        keys, values = kv[li, 0, :, :pos + 1], kv[li, 1, :, :pos + 1]
        scores = torch.matmul(q.view(KVH, H // KVH, dh), keys.transpose(1, 2).contiguous()) / math.sqrt(dh)
        x = x + lin(torch.matmul(torch.softmax(scores, dim=-1), values.contiguous()).reshape(1, H * dh), layer["o"])
        gate_up = lin(norm(x, layer["ln2"]), layer["gate_up"])
        x = x + lin(_silu(gate_up[:, :case["ffn"]]) * gate_up[:, case["ffn"]:], layer["down"])
    return lin(norm(x, model.norm), model.lm_head), kv


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        return _exact_linear(case, seed)
    if kind == "vecmat":
        a, b = _vecmat_inputs(case, seed)
        b = b.double()
        return a.double() @ (b.t().contiguous() if case["layout"] == "nk" else b)
    if kind == "weights":
        return _exact_weights(case, seed)
    return _exact_decode_step(case, seed)
