"""The work a user of this package has it do, as cases that can be timed and compared.

Every case goes through the public modules or launchers, the way a W8A8 inference program calls them:

  linear       one int8 linear (any of the epilogues)
  linear_set   the six linears of a decoder layer back to back: q, k, v, out, fc1 + GELU-quant, fc2
  layer        a whole decoder layer: a prompt, a chunk of a prompt, or a decode step against an int8 KV cache
  bmm_chain    attention from the stand-alone pieces: Q.K^T -> softmax -> P.V
  bmm_kn       P.V with V as it comes out of the projection, [keys, head_dim] (BMM_S8T_S8T_S8T)
  rows         the memory-bound row kernels around the linears
  dynamic      a linear whose fp activations are quantised on the fly

`listed()` are the sizes in common use, `draw(rng)` gives others of the same ranges.
"""
import math

import torch

from triton_int_amd.kernels.fused import (gelu_q, quantize_per_token_absmax,
                                          skip_layer_norm_fwd_fused_single_pass2, softmax_q)
from triton_int_amd.kernels.linear import linear_a8_w8_bfp32_ofp32
from triton_int_amd.nn.bmm import BMM_S8T_S8N_F32T, BMM_S8T_S8N_S8T, BMM_S8T_S8T_S8T
from triton_int_amd.nn.fused import DQ_Add_LayerNorm_Q, LayerNormQ, W8A8BFP32OFP32_GeLu_Q
from triton_int_amd.nn.linear import (DynamicW8A8BFP32OFP32Linear, W8A8B8O8Linear, W8A8B8O8LinearReLU,
                                      W8A8B32O32LinearWithoutScaling, W8A8BFP32OFP32Linear)
from triton_int_amd.nn.opt import W8A8OPTDecoderLayer

DEVICE = "cuda"
_HALF = {"fp16": torch.float16, "bf16": torch.bfloat16}

# the int8 linear modules by epilogue; fp16 / bf16 outputs come from the launcher with a bias of that type
_LINEARS = {"b8_o8": W8A8B8O8Linear, "b8_o8_relu": W8A8B8O8LinearReLU, "b32_o32": W8A8B32O32LinearWithoutScaling,
            "fp32": W8A8BFP32OFP32Linear, "gelu_q": W8A8BFP32OFP32_GeLu_Q}
_OUT_BYTES = {"b8_o8": 1, "b8_o8_relu": 1, "b32_o32": 4, "fp32": 4, "gelu_q": 1, "fp16": 2, "bf16": 2}

# (hidden, heads, ffn) of the decoder layers this repository builds: tests, 4096-wide linear set, default
_MODELS = ((1024, 8, 4096), (4096, 32, 16384), (5120, 40, 20480))


def listed():
    return [
        # a single small projection: all latency (the repository's first configuration)
        {"name": "linear_512x768x768", "kind": "linear", "epilogue": "b8_o8", "M": 512, "N": 768, "K": 768},
        # 64 sequences decoding together through one wide linear: a read of the weights (the M sweep's sizes)
        {"name": "linear_64x6848x10240_fp16", "kind": "linear", "epilogue": "fp16", "M": 64, "N": 6848, "K": 10240},
        # the headline linear set: 2048 prompt tokens through the linears of a 4096-wide layer
        {"name": "linear_set_2048x4096", "kind": "linear_set", "M": 2048, "hidden": 4096, "ffn": 16384},
        # a 2048-token prompt through a 5120-wide layer
        {"name": "prefill_1x2048_h5120", "kind": "layer", "model": 2, "B": 1, "S": 2048, "past": 0, "capacity": 0},
        # two prompts of the length text happens to have: no size a multiple of anything
        {"name": "prefill_2x333_h4096", "kind": "layer", "model": 1, "B": 2, "S": 333, "past": 0, "capacity": 0},
        # 64 more tokens of a prompt appended to the 1000 already cached (chunked prefill)
        {"name": "append_1x64_h4096", "kind": "layer", "model": 1, "B": 1, "S": 64, "past": 1000, "capacity": 2048},
        # one conversation, one token: position 1531 of a cache allocated for 2048
        {"name": "decode_1x1_h5120", "kind": "layer", "model": 2, "B": 1, "S": 1, "past": 1530, "capacity": 2048},
        # sixteen conversations decoding together, one token each
        {"name": "decode_16x1_h4096", "kind": "layer", "model": 1, "B": 16, "S": 1, "past": 1006, "capacity": 2048},
        # attention of 160 heads of 2048 x 2048 from the stand-alone BMMs and the softmax between them
        {"name": "bmm_chain_160x2048x128", "kind": "bmm_chain", "BH": 160, "S": 2048, "T": 2048, "D": 128, "causal": False},
        # P.V for V in row-major order, 40 heads
        {"name": "bmm_kn_40x1024x128", "kind": "bmm_kn", "BH": 40, "M": 1024, "K": 1024, "N": 128},
        # the row kernels between the linears, 8192 tokens of a 5120-wide model
        {"name": "rows_8192x5120_fp16", "kind": "rows", "rows": 8192, "cols": 5120, "dtype": "fp16"},
        # fp16 activations quantised per tensor on the way into the linear
        {"name": "dynamic_2000x5120_fp16", "kind": "dynamic", "M": 2000, "N": 5120, "K": 5120, "dtype": "fp16"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A matrix dimension: mostly a multiple of 16 as model widths are, now and then anything."""
    v = _log_int(rng, lo, hi)
    return v if rng.random() < 0.15 else max(16, v // 16 * 16)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear_set", "layer", "layer", "layer", "layer", "layer",
                       "bmm_chain", "bmm_kn", "rows", "dynamic"])
    if kind == "linear":
        while True:
            c = {"kind": kind, "epilogue": rng.choice(sorted(_OUT_BYTES)), "M": _log_int(rng, 1, 4096),
                 "N": _width(rng, 256, 20480), "K": _width(rng, 256, 20480)}
            if c["M"] * c["N"] * c["K"] <= 2048 * 5120 * 20480:
                return c
    if kind == "linear_set":
        hidden, _, ffn = rng.choice(_MODELS[:2])
        return {"kind": kind, "M": _log_int(rng, 1, 2048), "hidden": hidden, "ffn": ffn}
    if kind == "layer":
        model = rng.randrange(len(_MODELS))
        phase = rng.choice(["prefill", "append", "decode", "decode"])
        if phase == "prefill":
            B = rng.choice([1, 1, 2, 3, 4])
            S, past, capacity = _log_int(rng, 8, 2048 // B), 0, 0
        elif phase == "append":
            B, S, past = rng.choice([1, 1, 2]), _log_int(rng, 2, 256), _log_int(rng, 16, 1700)
            capacity = rng.choice([0, 2048])
        else:
            B, S, past, capacity = _log_int(rng, 1, 16), 1, _log_int(rng, 16, 2047), rng.choice([0, 2048, 2048])
        return {"kind": kind, "model": model, "B": B, "S": S, "past": past, "capacity": capacity}
    if kind == "bmm_chain":
        S = _log_int(rng, 16, 2048)
        return {"kind": kind, "BH": _log_int(rng, 8, 160), "S": S, "T": S, "D": rng.choice([64, 128, 128]), "causal": rng.random() < 0.5}
    if kind == "bmm_kn":
        S = _log_int(rng, 16, 2048)
        return {"kind": kind, "BH": _log_int(rng, 4, 80), "M": rng.choice([1, S, S, S]), "K": S, "N": rng.choice([64, 128, 128])}
    if kind == "rows":
        cols = _log_int(rng, 512, 8192)
        cols = cols if rng.random() < 0.15 else max(8, cols // 8 * 8)
        return {"kind": kind, "rows": _log_int(rng, 1, 8192 * 5120 // cols), "cols": cols, "dtype": rng.choice(["fp16", "bf16", "fp32"])}
    while True:
        c = {"kind": kind, "M": _log_int(rng, 1, 4096), "N": _log_int(rng, 256, 20480) // 16 * 16,
             "K": _log_int(rng, 256, 20480) // 16 * 16, "dtype": rng.choice(["fp16", "fp16", "fp32"])}
        if c["M"] * c["N"] * c["K"] <= 2048 * 5120 * 20480:
            return c


# ---- inputs -------------------------------------------------------------------------------------------

def _int8(g, shape, std=28.0):
    """Gaussian values quantised by their largest magnitude (about 4.5 sigma): what absmax quantisation gives."""
    return (torch.randn(shape, generator=g, device=DEVICE) * std).round_().clamp_(-127, 127).to(torch.int8)


def _scalar(v):
    return torch.tensor(v, dtype=torch.float32, device=DEVICE)


def _fill_linear(lin, g, a=None, b=None, bias_std=20.0):
    lin.weight = _int8(g, tuple(lin.weight.shape))
    n = lin.weight.shape[0]
    bias = torch.randn(n, generator=g, device=DEVICE) * bias_std
    lin.bias = bias.round().clamp(-127, 127).to(torch.int8) if lin.bias.dtype == torch.int8 else bias.to(lin.bias.dtype)
    if a is not None:
        lin.a = _scalar(a)
    if b is not None:
        lin.b = _scalar(b)
    return lin


def _make_linear(epilogue, N, K, g, x_std=28.0):
    """A linear whose outputs use their type's range: the accumulator's deviation is x_std * 28 * sqrt(K)."""
    acc = x_std * 28.0 * math.sqrt(K)
    with torch.device(DEVICE):
        lin = _LINEARS[epilogue](K, N)
    if epilogue in ("b8_o8", "b8_o8_relu"):
        return _fill_linear(lin, g, a=30.0 / acc, b=0.1)
    if epilogue == "b32_o32":
        return _fill_linear(lin, g, bias_std=1000.0)
    if epilogue == "fp32":
        return _fill_linear(lin, g, a=0.3 / acc, bias_std=0.1)
    return _fill_linear(lin, g, a=1.0 / acc, b=30.0, bias_std=0.1)


def _fill_norm(ln, g, output_scale=0.05):
    n = ln.weight.shape[0]
    ln.weight = (1.0 + 0.1 * torch.randn(n, generator=g, device=DEVICE)) / output_scale
    ln.bias = 0.1 * torch.randn(n, generator=g, device=DEVICE) / output_scale
    return ln


def _make_layer(case, g):
    hidden, heads, ffn = _MODELS[case["model"]]
    with torch.device(DEVICE):
        layer = W8A8OPTDecoderLayer(hidden, heads, ffn)
    _fill_norm(layer.ln1, g), _fill_norm(layer.ln2, g)  # int8 activations with a deviation of 20
    acc = 20.0 * 28.0 * math.sqrt(hidden)
    for lin in (layer.q_proj, layer.k_proj, layer.v_proj):
        _fill_linear(lin, g, a=30.0 / acc, b=0.1)
    _fill_linear(layer.out_proj, g, bias_std=1000.0)
    layer.ln2.input_scale = 0.3 / acc
    _fill_linear(layer.fc1, g, a=1.0 / acc, b=30.0, bias_std=0.1)
    _fill_linear(layer.fc2, g, a=0.3 / (20.0 * 28.0 * math.sqrt(ffn)), bias_std=0.1)
    # scores with a deviation of 25 steps, logits of 2.5
    layer.qk_alpha, layer.score_scale, layer.pv_alpha = 2.5e-3, 0.1, 0.05
    return layer


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "linear":
        M, N, K, epilogue = case["M"], case["N"], case["K"], case["epilogue"]
        s["x"] = _int8(g, (M, K))
        if epilogue in _HALF:
            s["w"] = _int8(g, (N, K))
            s["bias"] = (0.1 * torch.randn(N, generator=g, device=DEVICE)).to(_HALF[epilogue])
            s["a"], s["b"] = _scalar(0.3 / (28.0 * 28.0 * math.sqrt(K))), _scalar(1.0)
        else:
            s["linear"] = _make_linear(epilogue, N, K, g)
    elif kind == "linear_set":
        hidden, ffn = case["hidden"], case["ffn"]
        s["x"], s["f"] = _int8(g, (case["M"], hidden)), _int8(g, (case["M"], ffn))
        s["qkvo"] = [_make_linear("b8_o8", hidden, hidden, g) for _ in range(4)]
        s["fc1"], s["fc2"] = _make_linear("gelu_q", ffn, hidden, g), _make_linear("fp32", hidden, ffn, g)
    elif kind == "layer":
        hidden, heads, _ = _MODELS[case["model"]]
        B, S, past = case["B"], case["S"], case["past"]
        s["layer"] = _make_layer(case, g)
        s["x"] = torch.randn((B, S, hidden), generator=g, device=DEVICE)
        s["kv"] = None
        if past:
            # a cache allocated once for `capacity` positions and used as views of the current length
            # (0: allocated at the current length)
            T = past + S
            room = max(case["capacity"], T)
            k = _int8(g, (B * heads, room, hidden // heads), 30.0)
            vt = _int8(g, (B * heads, hidden // heads, room), 30.0)
            s["kv"] = (k[:, :T], vt[:, :, :T])
    elif kind == "bmm_chain":
        BH, S, T, D = case["BH"], case["S"], case["T"], case["D"]
        s["q"], s["k"], s["vt"] = _int8(g, (BH, S, D), 30.0), _int8(g, (BH, T, D), 30.0), _int8(g, (BH, D, T), 30.0)
        s["qk"] = BMM_S8T_S8N_S8T(25.0 / (900.0 * math.sqrt(D))).to(DEVICE)
        s["pv"] = BMM_S8T_S8N_F32T(1.0 / 127.0).to(DEVICE)
    elif kind == "bmm_kn":
        BH, M, K, N = case["BH"], case["M"], case["K"], case["N"]
        logits = 2.5 * torch.randn((BH, M, K), generator=g, device=DEVICE)
        s["p"] = logits.softmax(-1).mul_(127.0).round_().to(torch.int8)
        s["v"] = _int8(g, (BH, K, N), 30.0)
        s["bmm"] = BMM_S8T_S8T_S8T(0.05).to(DEVICE)
    elif kind == "rows":
        rows, cols = case["rows"], case["cols"]
        dtype = _HALF.get(case["dtype"], torch.float32)
        with torch.device(DEVICE):
            s["ln"], s["dq"] = LayerNormQ(cols), DQ_Add_LayerNorm_Q(cols)
        _fill_norm(s["ln"], g), _fill_norm(s["dq"], g)
        s["dq"].input_scale = 1e-5
        s["x"] = torch.randn((rows, cols), generator=g, device=DEVICE)
        s["acc"] = (torch.randn((rows, cols), generator=g, device=DEVICE) * 40000.0).to(torch.int32)
        s["gelu_scale"] = _scalar(30.0)
        s["h"] = torch.randn((rows, cols), generator=g, device=DEVICE).to(dtype)
        s["skip"] = torch.randn((rows, cols), generator=g, device=DEVICE).to(dtype)
        s["gamma"] = (1.0 + 0.1 * torch.randn(cols, generator=g, device=DEVICE)).to(dtype)
        s["beta"] = (0.1 * torch.randn(cols, generator=g, device=DEVICE)).to(dtype)
    else:
        with torch.device(DEVICE):
            lin = DynamicW8A8BFP32OFP32Linear(case["K"], case["N"])
        _fill_linear(lin, g, bias_std=0.1)
        lin.weight_scale = _scalar(1.0 / (28.0 * math.sqrt(case["K"])))
        s["linear"] = lin
        s["x"] = torch.randn((case["M"], case["K"]), generator=g, device=DEVICE).to(_HALF.get(case["dtype"], torch.float32))
    return s


# ---- one pass -----------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        if "w" in s:
            return linear_a8_w8_bfp32_ofp32(s["x"], s["w"], s["bias"], s["a"], s["b"])
        return s["linear"](s["x"])
    if kind == "linear_set":
        return [lin(s["x"]) for lin in s["qkvo"]] + [s["fc1"](s["x"]), s["fc2"](s["f"])]
    if kind == "layer":
        out = s["layer"](s["x"], kv_cache=s["kv"])
        return out if s["kv"] is None else (out, s["kv"][0], s["kv"][1])  # the caches are updated in place
    if kind == "bmm_chain":
        scores = s["qk"](s["q"], s["k"])
        probs = softmax_q(scores, 0.1, causal_q_len=case["S"] if case["causal"] else 0)
        return scores, probs, s["pv"](probs, s["vt"])
    if kind == "bmm_kn":
        return s["bmm"](s["p"], s["v"])
    if kind == "rows":
        h8 = s["ln"](s["x"])
        resid, y8 = s["dq"](s["x"], s["acc"])
        f8 = gelu_q(s["x"], s["gelu_scale"])
        normed, skipped = skip_layer_norm_fwd_fused_single_pass2(s["h"], s["skip"], s["gamma"], s["beta"], 1e-5)
        out = [h8, resid, y8, f8, normed, skipped]
        if s["h"].dtype != torch.bfloat16:
            out += quantize_per_token_absmax(s["h"])
        return out
    return s["linear"](s["x"])


# ---- what a pass cannot do without ----------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": M * K + N * K + M * N * _OUT_BYTES[case["epilogue"]] + 4 * N, "flops": 2 * M * N * K}
    if kind == "linear_set":
        M, H, F = case["M"], case["hidden"], case["ffn"]
        weights = 4 * H * H + 2 * H * F
        return {"bytes": weights + M * (H + F) + M * (4 * H + F + 4 * H), "flops": 2 * M * weights}
    if kind == "layer":
        H, _, F = _MODELS[case["model"]]
        B, S, past = case["B"], case["S"], case["past"]
        weights = 4 * H * H + 2 * H * F
        pairs = B * (S * past + S * (S + 1) // 2)  # (query, visible key), per head; D * heads = H
        return {"bytes": weights + 8 * B * S * H + 2 * B * H * past + (2 * B * H * S if past else 0),
                "flops": 2 * B * S * weights + 4 * pairs * H}
    if kind == "bmm_chain":
        BH, S, T, D = case["BH"], case["S"], case["T"], case["D"]
        # scores and probabilities are outputs; each is read once by the step after it
        return {"bytes": BH * (S * D + 2 * T * D + 4 * S * T + 4 * S * D), "flops": 4 * BH * S * T * D}
    if kind == "bmm_kn":
        BH, M, K, N = case["BH"], case["M"], case["K"], case["N"]
        return {"bytes": BH * (M * K + K * N + M * N), "flops": 2 * BH * M * N * K}
    if kind == "rows":
        n = case["rows"] * case["cols"]
        e = 4 if case["dtype"] == "fp32" else 2
        per = 5 + 13 + 5 + 4 * e + (e + 1 if case["dtype"] != "bf16" else 0)
        return {"bytes": n * per, "flops": 40 * n}
    M, N, K = case["M"], case["N"], case["K"]
    e = 4 if case["dtype"] == "fp32" else 2
    return {"bytes": M * K * e + N * K + 4 * M * N + 4 * N, "flops": 2 * M * N * K}


def tolerance(case):
    """Four times what each path shows against itself with the steps that depend on a summation order or on a
    transcendental function (LayerNorm, GELU, softmax) computed in 64 bits."""
    kind = case["kind"]
    if kind == "layer":  # int8 steps one apart early in the layer: rel 3.4e-3, max 0.10, caches differ in 2e-5
        return {"rel": 1.4e-2, "max": 0.4, "differ": 1e-4}
    if kind == "bmm_chain":  # rel 3.4e-4, 4.5e-8 of the probabilities one step apart (0 against 1)
        return {"rel": 1.4e-3, "max": 0.99, "differ": 1e-6}
    if kind in ("rows", "linear_set") or case.get("epilogue") == "gelu_q":  # rel 5.3e-5, 1.1e-6 one step apart
        return {"rel": 2e-4, "max": 0.2, "differ": 4e-6}
    return "exact"  # integer sums, with one rounding per fixed step before and after them
