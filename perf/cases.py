"""The work that a user of this package has it do, as timed cases.

Four kinds of case, each through the public entry points as an inference program calls them:

  layer   the projections of one or several transformer layers on device tensors: RMSNorm + quantizer, q / k / v, o,
          RMSNorm + quantizer, gate / up, SwiGLU + quantizer, down.  One token is decoding for one sequence, a few
          tokens are decoding for as many sequences at once, more are a prompt.  (Attention and the residual sums belong
          to the caller: its results are inputs here.)
  head    the vocabulary projection and the sampler behind it
  moe     a mixture-of-experts layer from router to weighted combine
  host    the projections of a layer through QuantLinear on host arrays, weights held by the weight cache
"""
import math

import numpy as np
import torch

from oxillama_amd import capi, linear, moe
from oxillama_amd.quant import GgufTensorType, KernelDispatcher, QuantTensor, quantize_q8_0_dev

TYPES = {"Q4_0": GgufTensorType.Q4_0, "Q5_0": GgufTensorType.Q5_0, "Q8_0": GgufTensorType.Q8_0,
         "IQ4_NL": GgufTensorType.Iq4Nl, "Q4_K": GgufTensorType.Q4K, "Q5_K": GgufTensorType.Q5K,
         "Q6_K": GgufTensorType.Q6K, "IQ4_XS": GgufTensorType.Iq4Xs}
EPS = 1e-5


# ---- cases ---------------------------------------------------------------------------------------------------


def _layer(tokens, hidden, kv, inter, attn, ffn, down, layers=1, bias=False):
    return {"kind": "layer", "tokens": tokens, "hidden": hidden, "kv": kv, "inter": inter, "attn": attn, "ffn": ffn,
            "down": down, "layers": layers, "bias": bias}


def _moe(tokens, experts, top_k, hidden, inter, ffn, down):
    return {"kind": "moe", "tokens": tokens, "experts": experts, "top_k": top_k, "hidden": hidden, "inter": inter,
            "ffn": ffn, "down": down}


def _head(vocab, hidden, wtype, greedy):
    return {"kind": "head", "vocab": vocab, "hidden": hidden, "wtype": wtype, "greedy": greedy}


def _host(hidden, kv, inter, attn, ffn, down):
    return {"kind": "host", "hidden": hidden, "kv": kv, "inter": inter, "attn": attn, "ffn": ffn, "down": down}


def listed():
    return [
        # one token through a layer of a small model (rows that are no multiple of 256, biases on q / k / v): the
        # smallest calls, all launch and host time
        dict(_layer(1, 896, 128, 4864, "Q8_0", "Q8_0", "Q8_0", bias=True), name="decode_1_small"),
        # interactive chat with an 8B model: one token through four layers whose weights come from HBM
        dict(_layer(1, 4096, 1024, 14336, "Q4_K", "Q4_K", "Q6_K", layers=4), name="decode_1_8b"),
        # a server's decode step for 16 sequences
        dict(_layer(16, 4096, 1024, 14336, "Q4_K", "Q4_K", "Q6_K"), name="decode_16_8b"),
        # a short chat prompt of odd length on a small model in a 32-weight format
        dict(_layer(77, 1536, 256, 8960, "Q4_0", "Q4_0", "Q8_0", bias=True), name="prompt_77_small"),
        # a prompt of odd length in the 5-bit files
        dict(_layer(333, 4096, 1024, 11008, "Q5_K", "Q5_K", "Q6_K"), name="prompt_333_q5k"),
        # the usual prompt chunk of an 8B model
        dict(_layer(512, 4096, 1024, 14336, "Q4_K", "Q4_K", "Q6_K"), name="prompt_512_8b"),
        # a long prompt on a layer of a 70B-class model
        dict(_layer(2048, 8192, 1024, 28672, "Q4_K", "Q4_K", "Q6_K"), name="prompt_2048_70b"),
        # the next token out of the last hidden state: logits, penalties, top-40, top-p, the draw
        dict(_head(128256, 4096, "Q6_K", False), name="head_sample"),
        # one token through eight large experts
        dict(_moe(1, 8, 2, 4096, 14336, "IQ4_XS", "IQ4_XS"), name="moe_1"),
        # a decode batch of 64 sequences through the same layer
        dict(_moe(64, 8, 2, 4096, 14336, "IQ4_XS", "IQ4_XS"), name="moe_64"),
        # a prompt chunk through many small experts
        dict(_moe(512, 128, 8, 2048, 768, "Q4_K", "Q6_K"), name="moe_512_small_experts"),
        # the kernel trait's host-slice route: one token, arrays in host memory in and out
        dict(_host(4096, 1024, 14336, "Q4_K", "Q4_K", "Q6_K"), name="host_1_8b"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _formats(rng, blocks_of_256):
    """(attention, feed-forward, down) formats as the usual files mix them."""
    if blocks_of_256:
        return rng.choice([("Q4_K", "Q4_K", "Q6_K"), ("Q4_K", "Q4_K", "Q4_K"), ("Q5_K", "Q5_K", "Q6_K"),
                           ("Q6_K", "Q6_K", "Q6_K"), ("IQ4_XS", "IQ4_XS", "IQ4_XS"), ("IQ4_XS", "IQ4_XS", "Q5_K"),
                           ("Q8_0", "Q8_0", "Q8_0"), ("Q4_0", "Q4_0", "Q4_0")])
    return rng.choice([("Q8_0", "Q8_0", "Q8_0"), ("Q4_0", "Q4_0", "Q4_0"), ("Q4_0", "Q4_0", "Q8_0"),
                       ("Q5_0", "Q5_0", "Q8_0"), ("IQ4_NL", "IQ4_NL", "IQ4_NL")])


def _dims(rng, most):
    """(hidden, kv, inter, whether rows are whole 256-weight blocks)"""
    whole = rng.random() < 0.7
    unit = 256 if whole else 32
    hidden = max(unit, round(_log_uniform(rng, 768, most) / unit) * unit)
    inter = round(hidden * rng.uniform(2.3, 5.8) / unit) * unit
    kv = max(128, hidden // rng.choice([1, 4, 8]) // 64 * 64)
    return hidden, kv, min(inter, 28672), whole


def draw(rng):
    u = rng.random()
    if u < 0.62:
        hidden, kv, inter, whole = _dims(rng, 8192)
        attn, ffn, down = _formats(rng, whole)
        tokens = 1 if rng.random() < 0.35 else max(2, round(_log_uniform(rng, 2, 2048)))
        layers = rng.choice([1, 2, 4]) if tokens == 1 else 1
        return _layer(tokens, hidden, kv, inter, attn, ffn, down, layers, rng.random() < 0.3)
    if u < 0.74:
        return _head(rng.randrange(32000, 152065), 256 * round(_log_uniform(rng, 4, 32)),
                     rng.choice(["Q6_K", "Q6_K", "Q8_0", "Q5_K"]), rng.random() < 0.4)
    if u < 0.9:
        tokens = 1 if rng.random() < 0.3 else max(2, round(_log_uniform(rng, 2, 512)))
        ffn, down = rng.choice([("IQ4_XS", "IQ4_XS"), ("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q5_K", "Q6_K"), ("Q4_0", "Q4_0")])
        if rng.random() < 0.5:
            return _moe(tokens, 8, 2, 256 * rng.randrange(8, 17), 256 * rng.randrange(24, 57), ffn, down)
        return _moe(tokens, rng.choice([32, 64, 128]), rng.choice([4, 6, 8]), 256 * rng.randrange(6, 13),
                    256 * rng.randrange(3, 7), ffn, down)
    hidden, kv, inter, whole = _dims(rng, 4096)
    return _host(hidden, kv, inter, *_formats(rng, whole))


# ---- inputs --------------------------------------------------------------------------------------------------


def _codes(gen, shape, lo, hi, mean, sd):
    """Quantized weights: normal weights rounded to the format's steps."""
    x = torch.randn(shape, generator=gen, device="cuda")
    return x.mul_(sd).add_(mean).round_().clamp_(lo, hi).to(torch.int16).to(torch.uint8)


def _half(gen, nb, scale):
    """Block scales as f16 bytes [nb, 2]: positive, spread by a quarter."""
    d = (torch.rand(nb, generator=gen, device="cuda") * 0.5 + 0.75) * scale
    return d.to(torch.float16).view(torch.uint8).view(nb, 2)


def _scales_6bit(gen, nb, zero_point):
    """Eight 6-bit scales and minima per block in the 12-byte packing of Q4_K and Q5_K; a minimum is near
    zero_point times its scale."""
    sc = torch.randint(30, 64, (nb, 8), generator=gen, device="cuda")
    mn = (sc + torch.randint(-4, 5, (nb, 8), generator=gen, device="cuda")).clamp_(0, 63) if zero_point else sc
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    return torch.cat([sc[:, :4] | (sc[:, 4:] >> 4) << 6, mn[:, :4] | (mn[:, 4:] >> 4) << 6,
                      (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4], 1)


def _weights(gen, wtype, rows, cols, sigma=0.02):
    """A matrix of normal weights as raw blocks of the format: uint8 [rows * row bytes] on the GPU."""
    t = TYPES[wtype]
    bs = t.block_size()
    nb = rows * (cols // bs)
    if wtype in ("Q4_0", "IQ4_NL"):
        q = _codes(gen, (nb, 32), 0, 15, 8.0, 2.7)
        parts = [_half(gen, nb, sigma / (2.7 if wtype == "Q4_0" else 45.0)), q[:, :16] | q[:, 16:] << 4]
    elif wtype == "Q5_0":
        q = _codes(gen, (nb, 32), 0, 31, 16.0, 5.5)
        bit = (q >> 4).view(nb, 4, 8) << torch.arange(8, device="cuda", dtype=torch.uint8)
        parts = [_half(gen, nb, sigma / 5.5), bit.sum(2, dtype=torch.int16).to(torch.uint8),
                 (q[:, :16] & 15) | (q[:, 16:] & 15) << 4]
    elif wtype == "Q8_0":
        q = torch.randn((nb, 32), generator=gen, device="cuda").mul_(48).round_().clamp_(-127, 127)
        parts = [_half(gen, nb, sigma / 48), q.to(torch.int8).view(torch.uint8)]
    elif wtype == "Q4_K":
        q = _codes(gen, (nb, 4, 2, 32), 0, 15, 7.5, 3.3)
        d = _half(gen, nb, sigma / (3.3 * 46))
        dmin = (d.view(torch.float16) * 7.5).view(torch.uint8)
        parts = [d, dmin, _scales_6bit(gen, nb, True), (q[:, :, 0] | q[:, :, 1] << 4).reshape(nb, 128)]
    elif wtype == "Q5_K":
        q = _codes(gen, (nb, 4, 2, 32), 0, 31, 15.5, 6.6)
        d = _half(gen, nb, sigma / (6.6 * 46))
        dmin = (d.view(torch.float16) * 15.5).view(torch.uint8)
        high = (q >> 4).view(nb, 8, 32) << torch.arange(8, device="cuda", dtype=torch.uint8).view(1, 8, 1)
        parts = [d, dmin, _scales_6bit(gen, nb, True), high.sum(1, dtype=torch.int16).to(torch.uint8),
                 ((q[:, :, 0] & 15) | (q[:, :, 1] & 15) << 4).reshape(nb, 128)]
    elif wtype == "Q6_K":
        q = _codes(gen, (nb, 2, 4, 32), 0, 63, 32.0, 11.0)
        low = torch.cat([(q[:, :, 0] & 15) | (q[:, :, 2] & 15) << 4, (q[:, :, 1] & 15) | (q[:, :, 3] & 15) << 4], 2)
        high = q[:, :, 0] >> 4 | (q[:, :, 1] >> 4) << 2 | (q[:, :, 2] >> 4) << 4 | (q[:, :, 3] >> 4) << 6
        sc = torch.randint(60, 128, (nb, 16), generator=gen, device="cuda") * (
            torch.randint(0, 2, (nb, 16), generator=gen, device="cuda") * 2 - 1)
        parts = [low.reshape(nb, 128), high.reshape(nb, 64), sc.to(torch.int8).view(torch.uint8), _half(gen, nb, sigma / (11 * 96))]
    elif wtype == "IQ4_XS":
        q = _codes(gen, (nb, 8, 32), 0, 15, 7.6, 2.7)
        ls = torch.randint(8, 57, (nb, 8), generator=gen, device="cuda")  # scale - 32 in -24..24
        high = ((ls >> 4) << (2 * torch.arange(8, device="cuda"))).sum(1).to(torch.int32)
        low = (ls[:, 0::2] & 15 | (ls[:, 1::2] & 15) << 4).to(torch.uint8)
        high = torch.stack([high & 255, high >> 8], 1).to(torch.uint8)
        parts = [_half(gen, nb, sigma / (45 * 13)), high, low, (q[:, :, :16] | q[:, :, 16:] << 4).reshape(nb, 128)]
    else:
        raise ValueError(wtype)
    w = torch.cat(parts, 1)
    assert w.shape[1] == t.block_bytes() and w.dtype == torch.uint8
    return w.view(-1)


def _acts(gen, *shape):
    """Activations: normal, a few columns much larger than the rest, as hidden states have them."""
    x = torch.randn(shape, generator=gen, device="cuda")
    x[..., :: max(1, shape[-1] // 5)] *= 6
    return x


def _f32(*shape):
    return torch.zeros(shape, device="cuda")


def _q8(n):
    return torch.zeros(n // 32 * 34, dtype=torch.uint8, device="cuda")


def _ws(nbytes):
    return torch.zeros(max(256, int(nbytes)), dtype=torch.uint8, device="cuda")


def _row_bytes(wtype, cols):
    t = TYPES[wtype]
    return cols // t.block_size() * t.block_bytes()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return {"layer": _prepare_layer, "head": _prepare_head, "moe": _prepare_moe, "host": _prepare_host}[case["kind"]](case, gen)


def _prepare_layer(case, gen):
    T, H, KV, I = case["tokens"], case["hidden"], case["kv"], case["inter"]
    shapes = {"q": (case["attn"], H, H), "k": (case["attn"], KV, H), "v": (case["attn"], KV, H), "o": (case["attn"], H, H),
              "gate": (case["ffn"], I, H), "up": (case["ffn"], I, H), "down": (case["down"], H, I)}
    ws = linear.ffn_workspace_bytes(H, I) if T == 1 else max(
        KernelDispatcher().get_kernel(TYPES[t]).gemm_workspace_bytes(T, n, k) for t, n, k in shapes.values())
    s = {"case": case, "ws": _ws(ws), "layers": []}
    for _ in range(case["layers"]):
        L = {name: _weights(gen, *sh) for name, sh in shapes.items()}
        L["norm1"], L["norm2"] = (1 + 0.1 * torch.randn(H, generator=gen, device="cuda") for _ in range(2))
        L["bias"] = [0.5 * torch.randn(n, generator=gen, device="cuda") for n in (H, KV, KV)] if case["bias"] else None
        L["x"], L["attn"], L["x2"] = (_acts(gen, T, H) for _ in range(3))
        L["q_out"], L["k_out"], L["v_out"], L["o_out"], L["y"] = (_f32(T, n) for n in (H, KV, KV, H, H))
        s["layers"].append(L)
    s["acts"], s["attn_q8"], s["acts2"] = _q8(T * H), _q8(T * H), _q8(T * H)
    if T > 1:
        s["gate_out"], s["up_out"], s["h_q8"] = _f32(T, I), _f32(T, I), _q8(T * I)
    return s


def _prepare_head(case, gen):
    V, H = case["vocab"], case["hidden"]
    k = 1 if case["greedy"] else 40
    t = TYPES[case["wtype"]]
    ws = linear.lm_head_topk_workspace_bytes(int(t), V, H, k) if case["greedy"] else linear.topk_workspace_bytes(V, k)
    return {"case": case, "t": t, "k": k, "w": _weights(gen, case["wtype"], V, H), "ws": _ws(ws),
            "norm": 1 + 0.1 * torch.randn(H, generator=gen, device="cuda"), "x": _acts(gen, 1, H), "acts": _q8(H),
            "logits": _f32(V), "values": _f32(k), "ids": torch.zeros(k, dtype=torch.int32, device="cuda"),
            "recent": torch.randint(0, V, (64,), generator=gen, device="cuda").to(torch.int32),
            "rng": torch.randint(1, 2**62, (1,), generator=gen, device="cuda"),
            "token": torch.zeros(1, dtype=torch.int32, device="cuda")}


def _prepare_moe(case, gen):
    T, E, H, I = case["tokens"], case["experts"], case["hidden"], case["inter"]
    tg, td = TYPES[case["ffn"]], TYPES[case["down"]]
    gate, up = ((tg, _weights(gen, case["ffn"], E * I, H), I * _row_bytes(case["ffn"], H)) for _ in range(2))
    down = (td, _weights(gen, case["down"], E * H, I), H * _row_bytes(case["down"], I))
    return {"case": case, "gate": gate, "up": up, "down": down, "x": _acts(gen, T, H),
            "router": torch.randn((E, H), generator=gen, device="cuda") / math.sqrt(H), "y": _f32(T, H),
            "ws": _ws(moe.moe_forward_workspace_bytes((tg, tg, td), T, case["top_k"], E, H, I))}


def _prepare_host(case, gen):
    H, KV, I = case["hidden"], case["kv"], case["inter"]
    capi.load().oxq_weight_cache_enable(1)  # as the binding does: weights do not change after loading
    s = []
    for wtype, n, k in ((case["attn"], H, H), (case["attn"], KV, H), (case["attn"], KV, H), (case["attn"], H, H),
                        (case["ffn"], I, H), (case["ffn"], I, H), (case["down"], H, I)):
        w = _weights(gen, wtype, n, k).cpu().numpy()
        s.append((linear.QuantLinear(QuantTensor(w, [n, k], TYPES[wtype])), KernelDispatcher().get_kernel(TYPES[wtype]),
                  _acts(gen, k).cpu().numpy(), np.zeros(n, np.float32)))
    return {"case": case, "linears": s}


# ---- one pass ------------------------------------------------------------------------------------------------


def run(state):
    kind = state["case"]["kind"]
    if kind == "layer":
        return _run_decode(state) if state["case"]["tokens"] == 1 else _run_batch(state)
    return {"head": _run_head, "moe": _run_moe, "host": _run_host}[kind](state)


def _run_decode(s):
    c = s["case"]
    H, KV, I = c["hidden"], c["kv"], c["inter"]
    attn, ffn, down = TYPES[c["attn"]], TYPES[c["ffn"]], TYPES[c["down"]]
    out = []
    for L in s["layers"]:
        linear.rmsnorm_quantize_dev(L["x"], L["norm1"], EPS, 1, H, d_out_q8=s["acts"])
        linear.linear_forward_multi_dev(attn, [L["q"], L["k"], L["v"]], s["acts"], [L["q_out"], L["k_out"], L["v_out"]],
                                        [H, KV, KV], H, L["bias"])
        linear.linear_forward_dev(attn, L["o"], L["o_out"], H, H, d_x=L["attn"])
        linear.rmsnorm_quantize_dev(L["x2"], L["norm2"], EPS, 1, H, d_out_q8=s["acts2"])
        linear.ffn_swiglu_dev((ffn, L["gate"]), (ffn, L["up"]), (down, L["down"]), s["acts2"], L["y"], H, I, s["ws"])
        out.append([L[name] for name in ("q_out", "k_out", "v_out", "o_out", "y")])
    return out


def _run_batch(s):
    c = s["case"]
    T, H, KV, I = c["tokens"], c["hidden"], c["kv"], c["inter"]
    attn, ffn, down = TYPES[c["attn"]], TYPES[c["ffn"]], TYPES[c["down"]]
    ws = s["ws"]
    out = []
    for L in s["layers"]:
        linear.rmsnorm_quantize_dev(L["x"], L["norm1"], EPS, T, H, d_out_q8=s["acts"])
        for i, (name, n) in enumerate((("q", H), ("k", KV), ("v", KV))):
            linear.linear_forward_batch_dev(attn, L[name], s["acts"], L[name + "_out"], T, n, H,
                                            d_bias=L["bias"][i] if L["bias"] else None, workspace=ws)
        quantize_q8_0_dev(L["attn"], s["attn_q8"])
        linear.linear_forward_batch_dev(attn, L["o"], s["attn_q8"], L["o_out"], T, H, H, workspace=ws)
        linear.rmsnorm_quantize_dev(L["x2"], L["norm2"], EPS, T, H, d_out_q8=s["acts2"])
        linear.linear_forward_batch_dev(ffn, L["gate"], s["acts2"], s["gate_out"], T, I, H, workspace=ws)
        linear.linear_forward_batch_dev(ffn, L["up"], s["acts2"], s["up_out"], T, I, H, workspace=ws)
        linear.swiglu_quantize_dev(s["gate_out"], s["up_out"], d_out_q8=s["h_q8"])
        linear.linear_forward_batch_dev(down, L["down"], s["h_q8"], L["y"], T, H, I, workspace=ws)
        out.append([L[name] for name in ("q_out", "k_out", "v_out", "o_out", "y")])
    return out


def _run_head(s):
    c = s["case"]
    V, H, k = c["vocab"], c["hidden"], s["k"]
    linear.rmsnorm_quantize_dev(s["x"], s["norm"], EPS, 1, H, d_out_q8=s["acts"])
    if c["greedy"]:
        linear.lm_head_topk_dev(int(s["t"]), s["w"], s["acts"], s["logits"], V, H, k, s["values"], s["ids"], s["ws"])
        return s["logits"], s["values"], s["ids"]
    linear.linear_forward_dev(s["t"], s["w"], s["logits"], V, H, d_acts=s["acts"])
    linear.logits_edit_dev(s["logits"], d_recent=s["recent"], window=64, repetition_penalty=1.1)
    linear.topk_dev(s["logits"], k, s["values"], s["ids"], s["ws"])
    linear.sample_candidates_dev(s["values"], s["ids"], k, 0.7, 0.0, 0.9, s["rng"], s["token"])
    return s["logits"], s["values"], s["ids"], s["token"], s["rng"]


def _run_moe(s):
    c = s["case"]
    moe.moe_forward_dev(s["gate"], s["up"], s["down"], c["experts"], s["router"], s["x"], c["tokens"], c["top_k"], s["y"],
                        c["hidden"], c["inter"], s["ws"])
    return s["y"]


def _run_host(s):
    for lin, kernel, x, out in s["linears"]:
        lin.forward(kernel, x, out)
    return [out for _, _, _, out in s["linears"]]


# ---- what a pass cannot do without ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "head":
        V, H = case["vocab"], case["hidden"]
        return {"bytes": V * _row_bytes(case["wtype"], H) + 8 * H + 4 * V, "flops": 2 * V * H}
    if kind == "moe":
        T, E, k, H, I = case["tokens"], case["experts"], case["top_k"], case["hidden"], case["inter"]
        used = E * (1 - (1 - k / E) ** T)  # experts that some token chooses, in the mean
        expert = 2 * I * _row_bytes(case["ffn"], H) + H * _row_bytes(case["down"], I)
        return {"bytes": used * expert + 4 * E * H + 8 * T * H, "flops": 2 * T * k * 3 * H * I + 2 * T * E * H}
    H, KV, I = case["hidden"], case["kv"], case["inter"]
    T, layers = case.get("tokens", 1), case.get("layers", 1)
    weights = (2 * H + 2 * KV) * _row_bytes(case["attn"], H) + 2 * I * _row_bytes(case["ffn"], H) + H * _row_bytes(case["down"], I)
    # the layer reads x, attention's result and x2 and writes q, k, v, o and y
    bytes_ = weights + 4 * T * (3 * H + 3 * H + 2 * KV)
    return {"bytes": layers * bytes_, "flops": layers * 2 * T * (2 * H * H + 2 * H * KV + 3 * H * I)}


def tolerance(case):
    # fp32 sums in another order (about 1e-6) move a few activations over a rounding boundary of the Q8_0 quantizer
    # between two stages; one such step is about 1/50 of an activation's root mean square, so a single one in a row of
    # 1000 to 5000 changes the row's product by 3e-4 to 6e-4 of its norm.
    if case["kind"] == "layer" or case["kind"] == "moe":
        return {"rel": 6e-4, "max": 1e-2}
    if case["kind"] == "head":
        return {"rel": 6e-4, "max": 1e-2, "differ": 0.0}
    return {"rel": 1e-5, "max": 1e-4}  # host: the same bytes in, fp32 sums of one product
