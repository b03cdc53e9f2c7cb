"""The work a user has this package do, as timed cases.

Every case is one pass through public entry points: a quantized linear as a drop-in module calls it
(`Int4Linear`, `AWQLinear`, `Int8Linear`, `Fp8Linear`, `MXFP4Linear`, `NVFP4Linear`, or the tiled
functions behind them for the asymmetric int4 format), the dynamic W8A8 linear, the quantizers a
checkpoint conversion or an FP8 KV cache runs, and the int4 decode step of a Llama-shaped model as a
captured graph. Sizes are those of the Llama-3-8B layers (4096 -> 1024 / 4096 / 14336 / 28672 and
14336 -> 4096) and the Llama-3-70B MLP (8192 <-> 28672) that `bench.py` names; prompts are ragged
where a server's are.

`listed()` holds the named cases; `draw(rng)` gives others of the same ranges: 1 row to a prompt of
2048 (4096 for MXFP4 x MXFP4), widths from 512 up, odd ones among them, with and without a bias, in
the activation types each linear takes.
"""

from __future__ import annotations

import math

import torch

from scratch_llm_amd import decode
from scratch_llm_amd.quant import awq, fp8_kv_per_head, fp8_weights, int4_group, int8, modules, nvfp4_mxfp4

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
GROUP = 128
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
FP8_MIN_SCALE = 1.0 / (448.0 * 512.0)

# the decode model: Llama-3-8B's layer and vocabulary, four layers deep
LAYERS, D, HEADS, KV_HEADS, HEAD_DIM, D_FF, VOCAB = 4, 4096, 32, 8, 128, 14336, 128256


def listed():
    return [
        # one token through the smallest projection (k or v of a GQA layer): launch latency and host cost
        {"name": "int4_asym_row", "kind": "int4", "m": 1, "n": 1024, "k": 4096, "asym": True, "dtype": "bf16",
         "bias": False},
        # a small continuous batch through the gate|up projection of AWQ weights
        {"name": "awq_batch", "kind": "awq", "m": 24, "n": 28672, "k": 4096, "dtype": "bf16", "bias": False},
        # a long prompt through the up projection of AWQ weights
        {"name": "awq_prompt", "kind": "awq", "m": 2048, "n": 14336, "k": 4096, "dtype": "bf16", "bias": False},
        # a short ragged prompt through an int8 weight-only projection with a bias
        {"name": "int8_prompt", "kind": "int8", "m": 500, "n": 4096, "k": 4096, "dtype": "bf16", "bias": True},
        # a batch of sixteen streams through the FP8 gate|up projection
        {"name": "fp8_batch", "kind": "fp8", "m": 16, "n": 28672, "k": 4096, "dtype": "bf16", "bias": False},
        # a prompt through the FP8 down projection
        {"name": "fp8_prompt", "kind": "fp8", "m": 1000, "n": 4096, "k": 14336, "dtype": "bf16", "bias": False},
        # a decode batch through the 70B up projection, MXFP4 weights and bf16 activations
        {"name": "mxfp4_batch", "kind": "mxfp4", "m": 32, "n": 28672, "k": 8192, "dtype": "bf16", "bias": False},
        # a long prompt through the 70B up projection with both operands in MXFP4: the largest call
        {"name": "mxfp4_act_prompt", "kind": "mxfp4_act", "m": 4096, "n": 28672, "k": 8192, "dtype": "bf16",
         "bias": False},
        # the dynamic W8A8 linear: both operands quantized in the call
        {"name": "w8a8_call", "kind": "w8a8", "m": 256, "n": 4096, "k": 4096, "dtype": "bf16"},
        # converting one checkpoint weight to int4 at load time
        {"name": "quantize_int4", "kind": "quantize", "fmt": "int4", "m": 14336, "k": 4096, "dtype": "bf16"},
        # a decode step of eight streams over a bf16 KV cache
        {"name": "decode_b8", "kind": "decode", "b": 8, "ctx": 2048, "kv": "bf16"},
        # a decode step of sixty-four streams over an FP8 KV cache
        {"name": "decode_b64_fp8kv", "kind": "decode", "b": 64, "ctx": 2048, "kv": "fp8"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["int4", "awq", "int8", "fp8", "mxfp4", "nvfp4", "mxfp4_act", "w8a8", "quantize", "decode"])
    if kind == "decode":
        return {"kind": kind, "b": _log_int(rng, 1, 64), "ctx": rng.choice([512, 1024, 2048]),
                "kv": rng.choice(["bf16", "fp8"])}
    if kind == "quantize":
        fmt = rng.choice(["int4", "int8", "fp8", "mxfp4", "nvfp4", "kv"])
        m = _log_int(rng, 128, 14336)
        return {"kind": kind, "fmt": fmt, "m": m, "k": 128 * _log_int(rng, 8, max(8, min(112, 14336 * 32 // m))),
                "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    k = 128 * _log_int(rng, 4, 112)
    if kind in ("int8", "fp8", "w8a8") and rng.random() < 0.3:
        k -= 16 * rng.randint(1, 7)
    elif kind in ("mxfp4", "mxfp4_act") and rng.random() < 0.3:
        k -= 32 * rng.randint(1, 3)
    n = _log_int(rng, 512, 28672)
    if rng.random() < 0.7:
        n = max(512, n // 16 * 16)
    cap = 4096 * 28672 * 8192 if kind == "mxfp4_act" else 2048 * 14336 * 4096
    m = min(_log_int(rng, 1, 4096 if kind == "mxfp4_act" else 2048), max(1, cap // (n * k)))
    case = {"kind": kind, "m": m, "n": n, "k": k, "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16"])}
    if kind == "w8a8":
        case["dtype"] = rng.choice(["bf16", "fp32"])
        return case
    case["bias"] = rng.random() < 0.3
    if kind == "mxfp4_act":
        case["dtype"] = "bf16"
    if kind == "int4":
        case["asym"] = rng.random() < 0.3
    if kind in ("int4", "awq") and not case.get("asym") and rng.random() < 0.15:
        case["dtype"], case["m"] = "fp32", min(m, 256)
    return case


# ----------------------------------------------------------------------------------------------
# Inputs, from the seed alone. Weights are drawn as a checkpoint holds them: integer codes and their
# scales (a quantized normal weight fills its code range), activations ~N(0, 1).
# ----------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _randint(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi, shape, device="cuda", generator=g, dtype=dtype)


def _group_scales(g, n, groups):
    """Scales of int4 groups of a N(0, 0.02) weight: absmax over 128 values / 7, spread by a few percent."""
    return 0.0075 * (1.0 + 0.1 * _randn(g, n, groups)).clamp_(0.5, 1.5)


def _linear_inputs(case, seed):
    """x, bias and the weight's stored tensors of one linear case."""
    g = _gen(seed)
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    dt = DTYPES[case["dtype"]]
    out = {"x": _randn(g, m, k).to(dt), "bias": (0.1 * _randn(g, n)).to(dt) if case.get("bias") else None}
    if kind in ("int4", "awq"):
        out["s"] = _group_scales(g, n, k // GROUP)
        if case.get("asym"):
            out["q"] = _randint(g, 0, 16, (n, k), torch.uint8)
            out["s"] = (out["s"] * (14.0 / 15.0)).to(torch.bfloat16)
            out["z"] = _randint(g, 5, 11, (n, k // GROUP), torch.int32).to(torch.bfloat16)
        else:
            out["q"] = (3.0 * _randn(g, n, k)).round_().clamp_(-7, 7).to(torch.int8)
        if kind == "awq":
            out["chan"] = torch.exp(0.4 * _randn(g, k))
    elif kind == "int8":
        out["q"] = (32.0 * _randn(g, n, k)).round_().clamp_(-127, 127).to(torch.int8)
        out["s"] = 0.0006 * (1.0 + 0.1 * _randn(g, n, 1)).clamp_(0.5, 1.5)
    elif kind == "fp8":
        out["q"] = (110.0 * _randn(g, n, k)).clamp_(-448, 448).to(torch.float8_e4m3fn)
        out["s"] = 0.00018 * (1.0 + 0.1 * _randn(g, n, 1)).clamp_(0.5, 1.5)
    elif kind in ("mxfp4", "mxfp4_act"):
        out["q"] = _randint(g, 0, 256, (n, k // 2), torch.uint8)
        out["s"] = _randint(g, 119, 123, (n, k // 32), torch.uint8)  # E8M0: 2**-8 .. 2**-5
    elif kind == "nvfp4":
        out["q"] = _randint(g, 0, 16, (n * k // 16, 16), torch.uint8)
        out["s"] = (0.5 * (1.0 + 6.0 * torch.rand(n * k // 16, device="cuda", generator=g))).to(torch.float8_e4m3fn).float()
        out["g"] = torch.full((), 0.004, device="cuda")
    elif kind == "w8a8":
        out["w"] = (0.02 * _randn(g, n, k)).to(dt)
    return out


def _kv_block(case, g):
    """A block of keys [1, 8, tokens, 128] for the FP8 cache: as many elements as the [m, k] matrix."""
    tokens = max(1, case["m"] * case["k"] // (KV_HEADS * HEAD_DIM))
    return _randn(g, 1, KV_HEADS, tokens, HEAD_DIM).to(DTYPES[case["dtype"]])


def _quantize_input(case, seed):
    g = _gen(seed)
    if case["fmt"] == "kv":
        return _kv_block(case, g)
    return (0.02 * _randn(g, case["m"], case["k"])).to(DTYPES[case["dtype"]])


_SHAPES = {
    "attn.q_proj": (HEADS * HEAD_DIM, D), "attn.k_proj": (KV_HEADS * HEAD_DIM, D), "attn.v_proj": (KV_HEADS * HEAD_DIM, D),
    "attn.o_proj": (D, HEADS * HEAD_DIM), "ffn.w1": (D_FF, D), "ffn.w3": (D_FF, D), "ffn.w2": (D, D_FF),
}
_NAMES = ["token_emb", "final_norm", "lm_head"] + [
    f"blocks.{i}.{p}" for i in range(LAYERS) for p in ("attn_norm", "ffn_norm", *_SHAPES)]


def _model_tensor(name, seed):
    """A float parameter of the decode model by its state-dict name (without ".weight")."""
    g = _gen(seed * 1009 + 1 + _NAMES.index(name))
    if name.endswith("norm"):
        return (1.0 + 0.1 * _randn(g, D)).to(torch.bfloat16).float()
    if name == "token_emb":
        return _randn(g, VOCAB, D).to(torch.bfloat16)
    shape = (VOCAB, D) if name == "lm_head" else _SHAPES[name.split(".", 2)[2]]
    return 0.02 * _randn(g, *shape)


def _decode_inputs(case, seed):
    """tokens, lengths, and a function giving layer i's cached keys and values [B, Hkv, ctx, 128]."""
    g = _gen(seed * 1009 + 7)
    b, ctx = case["b"], case["ctx"]
    tokens = _randint(g, 0, VOCAB, (b,), torch.int32)
    lengths = _randint(g, ctx // 2, ctx - 1, (b,), torch.int32)

    def kv(i):
        gi = _gen(seed * 1009 + 500 + i)
        return tuple(_randn(gi, b, KV_HEADS, ctx, HEAD_DIM).to(torch.bfloat16) for _ in range(2))

    return tokens, lengths, kv


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        cfg = decode.DecodeConfig(vocab_size=VOCAB, d_model=D, n_layers=LAYERS, n_heads=HEADS, n_kv_heads=KV_HEADS,
                                  d_ff=D_FF, context_length=2048)
        model = decode.Int4DecodeLM.from_state_dict(
            cfg, lambda name: _model_tensor(name.removesuffix(".weight"), seed), "cuda")
        state = model.new_state(case["b"], case["ctx"], kv_dtype=case["kv"])
        tokens, lengths, kv = _decode_inputs(case, seed)
        for i in range(LAYERS):
            k, v = kv(i)
            if case["kv"] == "fp8":
                state.set_kv_scales(i, fp8_kv_per_head.per_head_scale(k), fp8_kv_per_head.per_head_scale(v))
            state.write_kv(i, k, v)
        state.tokens.copy_(tokens)
        state.lengths.copy_(lengths)
        graph = model.capture(state)
        return {"kind": kind, "model": model, "state": state, "graph": graph, "tokens": tokens, "lengths": lengths}
    if kind == "quantize":
        return {"kind": kind, "fmt": case["fmt"], "w": _quantize_input(case, seed)}
    t = _linear_inputs(case, seed)
    x, q, s, bias, n, k = t["x"], t.get("q"), t.get("s"), t["bias"], case["n"], case["k"]
    if kind == "w8a8":
        return {"kind": kind, "x": x, "w": t["w"]}
    if kind == "int4" and case["asym"]:
        return {"kind": "int4_asym", "x": x, "tiled": int4_group.tile_int4(q, s, t["z"], GROUP), "bias": bias}
    if kind == "int4" and case["dtype"] == "fp32":
        return {"kind": "int4_codes", "x": x, "q": q, "s": s, "bias": bias}
    if kind == "int4":
        layer = modules.Int4Linear(int4_group.pack_int4(q.reshape(-1)), s, bias, k, n, GROUP)
    elif kind == "awq":
        layer = modules.AWQLinear(awq.AWQQuant(q=q, group_scales=s, chan_scale=t["chan"], group_size=GROUP), bias)
    elif kind == "int8":
        layer = modules.Int8Linear(q, s, bias)
    elif kind == "fp8":
        layer = fp8_weights.Fp8Linear(q, s, bias, out_dtype=DTYPES[case["dtype"]])
    elif kind == "nvfp4":
        layer = modules.NVFP4Linear(nvfp4_mxfp4.NVFP4Tensor(q, t["g"], s, torch.Size((n, k)), n * k, 16), bias)
    else:
        layer = modules.MXFP4Linear(q, s, bias, quantize_activations=kind == "mxfp4_act")
    return {"kind": kind, "x": x, "layer": layer}


def run(state):
    kind = state["kind"]
    if kind == "decode":
        st = state["state"]
        # a server writes the step's tokens and positions into the slots, then replays
        st.tokens.copy_(state["tokens"])
        st.lengths.copy_(state["lengths"])
        state["graph"].replay()
        return {"logits": st.logits, "tokens": st.tokens, "lengths": st.lengths, "k": st.k, "v": st.v}
    if kind == "quantize":
        w, fmt = state["w"], state["fmt"]
        if fmt == "int4":
            return int4_group.quantize_groupwise_int4(w, GROUP)
        if fmt == "int8":
            return int8.quantize_symmetric(w, axis=0)
        if fmt == "fp8":
            return fp8_weights.quantize_per_channel(w)
        if fmt == "kv":
            scale = fp8_kv_per_head.per_head_scale(w)
            return fp8_kv_per_head.quantize_per_head(w, scale), scale
        if fmt == "mxfp4":
            t = nvfp4_mxfp4.mxfp4_quantize(w)
            return t.codes, t.s_block
        t = nvfp4_mxfp4.nvfp4_quantize(w)
        return t.codes, t.s_block, t.s_global
    if kind == "w8a8":
        return int8.w8a8_linear(state["x"], state["w"])
    if kind == "int4_asym":
        return int4_group.int4_linear_tiled(state["x"], state["tiled"], state["bias"])
    if kind == "int4_codes":
        return int4_group.w4a16_linear(state["x"], state["q"], state["s"], state["bias"], GROUP)
    return state["layer"](state["x"])


# bytes of one stored weight, codes and scales
_WEIGHT_BYTES = {"awq": 0.5 + 4 / GROUP, "int8": 1.0, "fp8": 1.0, "mxfp4": 0.5 + 1 / 32, "mxfp4_act": 0.5 + 1 / 32,
                 "nvfp4": 0.5 + 1 / 16}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        layer = sum(a * b for a, b in _SHAPES.values())
        weights = LAYERS * layer + VOCAB * D
        kv = 2 * LAYERS * case["b"] * KV_HEADS * (3 * case["ctx"] // 4) * HEAD_DIM  # mean length: 3/4 of the context
        return {"bytes": weights * (0.5 + 4 / GROUP) + kv * (1 if case["kv"] == "fp8" else 2) + 2 * case["b"] * VOCAB,
                "flops": 2 * case["b"] * weights + 2 * kv * (HEADS // KV_HEADS)}
    es = 4 if case["dtype"] == "fp32" else 2
    if kind == "quantize":
        n = case["m"] * case["k"]
        out = {"int4": 1 + 4 / GROUP, "int8": 1, "fp8": 1, "kv": 1, "mxfp4": 1 + 4 / 32, "nvfp4": 1 + 4 / 16}[case["fmt"]]
        return {"bytes": n * (es + out), "flops": 2 * n}
    m, n, k = case["m"], case["n"], case["k"]
    if kind == "w8a8":
        return {"bytes": es * (m + n) * k + 4 * m * n, "flops": 2 * m * n * k}
    wb = 0.5 + 4 / GROUP if kind == "int4" else _WEIGHT_BYTES[kind]
    return {"bytes": wb * n * k + es * m * (k + n), "flops": 2 * m * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "decode":
        # bf16 roundings of one sub-layer travel through all that follow (1.1e-2 from the 64-bit logits after four
        # layers); near-tied logits may swap the pick, and a code of the new FP8 key or value may round the other way
        return {"rel": 4e-2, "max": 0.25, "differ": 0.02}
    if kind == "w8a8":
        return {"rel": 1e-6, "max": 1e-5}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    # 16-bit outputs: one rounding of the result, and in the prompt forms one of each dequantized weight
    # (measured against 64 bits: bf16 1.7e-3 to 2.8e-3, fp16 2.9e-4)
    return {"rel": 1e-2, "max": 6e-2} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 1e-2}


# ----------------------------------------------------------------------------------------------
# The same results in 64 bits, in plain torch
# ----------------------------------------------------------------------------------------------
def _rows_matmul(x, w_rows, n, chunk=4096):
    """x [m, k] times the rows of the weight, dequantized chunk by chunk to float64."""
    return torch.cat([x @ w_rows(i, min(n, i + chunk)).t() for i in range(0, n, chunk)], dim=1)


def _e2m1(codes):
    lut = torch.tensor(E2M1 + tuple(-v for v in E2M1), device=codes.device, dtype=torch.float64)
    return lut[codes.long()]


def _mxfp4_values(x):
    """The MXFP4 quantization of each row of x in blocks of 32, as float64 values (ties toward zero)."""
    xf = x.float()
    m, k = xf.shape
    b = xf.reshape(m, k // 32, 32)
    amax = b.abs().amax(dim=2, keepdim=True)
    scale = torch.exp2(torch.ceil(torch.log2((amax.double() / 6.0).clamp_min(1e-30))))
    mags = (b.double() / scale).abs()
    mid = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=x.device, dtype=torch.float64)
    vals = torch.tensor(E2M1, device=x.device, dtype=torch.float64)[torch.searchsorted(mid, mags.contiguous())]
    return (torch.sign(b.double()) * vals * scale).reshape(m, k)


def _int8_rows(x):
    """Symmetric int8 rows computed in x's dtype, as float64 codes and the scale in that dtype."""
    s = (x.abs().amax(dim=1, keepdim=True) / 127).clamp_min(1e-12)
    return (x / s).round().clamp(-127, 127).double(), s


def _fp8(x, s):
    return (x.float() / s).clamp(-448, 448).to(torch.float8_e4m3fn)


def _int4_weight(name, seed):
    """The int4 group-128 weight of a model tensor, as float64."""
    w = _model_tensor(name, seed)
    n, k = w.shape
    out = torch.empty(n, k, dtype=torch.float64, device=w.device)
    for i in range(0, n, 16384):
        g = w[i:i + 16384].reshape(-1, k // GROUP, GROUP)
        s = (g.abs().amax(dim=2, keepdim=True) / 7).clamp_min(torch.finfo(torch.float32).tiny)
        out[i:i + 16384] = ((g / s).round().clamp(-8, 7).double() * s.double()).reshape(-1, k)
    return out


def _rms(x, gain):
    return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + 1e-5) * gain.double()


def _exact_decode(case, seed):
    b, ctx = case["b"], case["ctx"]
    tokens, lengths, kv = _decode_inputs(case, seed)
    rows, pos = torch.arange(b, device="cuda"), lengths.long()
    inv = 1.0 / (10000.0 ** (torch.arange(0, HEAD_DIM, 2).float() / HEAD_DIM))
    angles = torch.outer(torch.arange(2048).float(), inv)
    cos, sin = (t.to("cuda")[pos].double()[:, None] for t in (angles.cos(), angles.sin()))

    def rope(t):  # [B, heads, 128], rotated in interleaved pairs
        e, o = t[..., 0::2], t[..., 1::2]
        return torch.stack((e * cos - o * sin, e * sin + o * cos), dim=-1).flatten(-2)

    seen = torch.arange(ctx, device="cuda")[None] <= pos[:, None]
    x = _model_tensor("token_emb", seed)[tokens.long()].double()
    k_out, v_out = [], []
    for i in range(LAYERS):
        p = f"blocks.{i}."
        h = _rms(x, _model_tensor(p + "attn_norm", seed))
        q, kn, vn = ((h @ _int4_weight(p + f"attn.{c}_proj", seed).t()).reshape(b, -1, HEAD_DIM) for c in "qkv")
        new = rope(kn), vn
        cache = []
        for old, fresh in zip(kv(i), new):
            if case["kv"] == "fp8":
                s = (old.float().abs().amax(dim=(0, 2, 3)) / 448).clamp_min(FP8_MIN_SCALE)
                old = _fp8(old, s.view(1, -1, 1, 1)).double() * s.double().view(1, -1, 1, 1)
                fresh = _fp8(fresh, s.view(1, -1, 1)).double() * s.double().view(1, -1, 1)
            t = old.double()
            t[rows, :, pos] = fresh
            cache.append(t)
        k, v = cache
        qg = rope(q).reshape(b, KV_HEADS, HEADS // KV_HEADS, HEAD_DIM)
        att = torch.empty(b, KV_HEADS, HEADS // KV_HEADS, HEAD_DIM, dtype=torch.float64, device="cuda")
        for r in range(b):
            score = (qg[r] @ k[r].transpose(1, 2).contiguous()) / math.sqrt(HEAD_DIM)
            att[r] = torch.softmax(score.masked_fill(~seen[r], float("-inf")), dim=-1) @ v[r]
        x = x + att.reshape(b, -1) @ _int4_weight(p + "attn.o_proj", seed).t()
        h = _rms(x, _model_tensor(p + "ffn_norm", seed))
        gate = h @ _int4_weight(p + "ffn.w1", seed).t()
        up = h @ _int4_weight(p + "ffn.w3", seed).t()
        x = x + (gate * torch.sigmoid(gate) * up) @ _int4_weight(p + "ffn.w2", seed).t()
        if case["kv"] == "bf16":
            k_out.append(k)
            v_out.append(v)
    logits = _rms(x, _model_tensor("final_norm", seed)) @ _int4_weight("lm_head", seed).t()
    full = case["kv"] == "bf16"
    return {"logits": logits, "tokens": None, "lengths": None, "k": torch.stack(k_out) if full else None,
            "v": torch.stack(v_out) if full else None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _exact_decode(case, seed)
    if kind == "quantize":
        return None
    t = _linear_inputs(case, seed)
    x, q, s, n, k = t["x"], t.get("q"), t.get("s"), case["n"], case["k"]
    if kind == "w8a8":
        qx, sx = _int8_rows(x)
        qw, sw = _int8_rows(t["w"])
        return (qx @ qw.t()) * (sx * sw.t()).double()
    xd = x.double()
    if kind in ("int4", "awq"):
        if kind == "awq":
            xd = xd / t["chan"].double()
        z = t["z"].double() if case.get("asym") else torch.zeros((n, k // GROUP), dtype=torch.float64, device="cuda")

        def rows(a, b):
            w = q[a:b].double().reshape(b - a, k // GROUP, GROUP) - z[a:b, :, None]
            return (w * s[a:b].double()[:, :, None]).reshape(b - a, k)
    elif kind in ("int8", "fp8"):
        if kind == "fp8":
            xf = x.float()
            sx = (xf.abs().amax(dim=1, keepdim=True) / 448).clamp_min(FP8_MIN_SCALE)
            xd = _fp8(xf, sx).double() * sx.double()

        def rows(a, b):
            return q[a:b].double() * s[a:b].double()
    elif kind == "nvfp4":
        def rows(a, b):
            blk = slice(a * k // 16, b * k // 16)
            return (_e2m1(q[blk]) * s[blk].double()[:, None] * t["g"].double()).reshape(b - a, k)
    else:
        if kind == "mxfp4_act":
            xd = _mxfp4_values(x)

        def rows(a, b):
            codes = torch.stack((q[a:b] & 15, q[a:b] >> 4), dim=2).reshape(b - a, k // 32, 32)
            return (_e2m1(codes) * torch.exp2(s[a:b].double() - 127.0)[:, :, None]).reshape(b - a, k)
    y = _rows_matmul(xd, rows, n)
    return y if t["bias"] is None else y + t["bias"].double()
