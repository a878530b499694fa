"""Performance cases of the quantized-contraction operators, through ``intent_amd.compile``.

Each case is one call (or the short chain of calls) that a program serving or
evaluating a quantized transformer makes per layer: weight-only int8 / int4
projections, int8 x int8 projections behind the per-token quantizer, block-scaled
FP8 projections behind the groupwise quantizer, a GGUF Q4_K projection and the two
mixture-of-experts feed-forward layers, at decode, at small ragged batches and at
prefill. ``draw`` samples the same families over the ranges given beside each
``_draw_*`` function.

Weights follow the distributions of ``intent_amd.inputs`` (uniform nibbles and int8,
uniform scales, N(0, 1) activations and logits), drawn on the GPU from the seed.
"""
import torch

import intent_amd as intent

_ARTIFACTS = {}


def _artifact(definition, **constexprs):
    """The compiled operator a program keeps for its lifetime."""
    key = (definition.name, tuple(sorted(constexprs.items())))
    if key not in _ARTIFACTS:
        _ARTIFACTS[key] = intent.compile(definition, target=intent.MI355XTarget(0), constexprs=constexprs or None)
    return _ARTIFACTS[key]


def listed():
    return [
        # the smallest call: a narrow int8 projection for a batch of 16 sequences
        {"name": "w8a16_m16_1k", "family": "w8a16", "M": 16, "K": 1024, "N": 1024, "prepared": False},
        # one sequence decoding: the attention output projection, bound once and launched per token
        {"name": "w4a16_decode_m1", "family": "w4a16", "M": 1, "K": 4096, "N": 4096, "group": 128, "prepared": True},
        # a dozen sequences decoding: the MLP up projection
        {"name": "w4a16_decode_m12", "family": "w4a16", "M": 12, "K": 4096, "N": 11008, "group": 128,
         "prepared": False},
        # a short prompt, or a large decode batch, of odd length
        {"name": "w4a16_batch_m77", "family": "w4a16", "M": 77, "K": 4096, "N": 4096, "group": 128, "prepared": False},
        # prefill of 2048 tokens through the MLP up projection
        {"name": "w4a16_prefill_m2048", "family": "w4a16", "M": 2048, "K": 4096, "N": 11008, "group": 128,
         "prepared": False},
        # int8 x int8 for a decode batch: per-token quantizer, then the projection
        {"name": "w8a8_decode_m32", "family": "w8a8", "M": 32, "K": 8192, "N": 8192},
        # the same for a 4096-token prefill
        {"name": "w8a8_prefill_m4096", "family": "w8a8", "M": 4096, "K": 8192, "N": 8192},
        # the W4 mixture-of-experts layer for 16 decoding sequences, and for a 512-token chunk
        {"name": "moe_w4_decode_t16", "family": "moe_w4", "T": 16, "H": 4096, "F": 14336, "E": 8, "top_k": 2,
         "group": 128},
        {"name": "moe_w4_chunk_t512", "family": "moe_w4", "T": 512, "H": 4096, "F": 14336, "E": 8, "top_k": 2,
         "group": 128},
        # the float mixture-of-experts layer over ragged routes, for 200 tokens
        {"name": "moe_f16_t200", "family": "moe_f16", "T": 200, "D": 4096, "F": 14336, "E": 8, "top_k": 2},
        # block-scaled FP8 for a ragged chunk: groupwise quantizer, then the MLP up projection
        {"name": "fp8_block_m300", "family": "fp8_block", "M": 300, "K": 4096, "N": 14336},
        # one sequence decoding through a GGUF Q4_K down projection
        {"name": "q4k_down", "family": "q4k", "K": 14336, "N": 4096},
    ]


# ---- drawn cases -----------------------------------------------------------------------

def _log_int(rng, low, high):
    return min(high, int(low * (high / low) ** rng.random() + 0.5))


def _rows(rng, high, flops_per_row, budget):
    """Rows over the logarithm of 1..high, within a budget of operations."""
    return _log_int(rng, 1, max(1, min(high, int(budget / flops_per_row))))


def _width(rng, low, high):
    """Output columns: whole 64s three times in four, any number (a vocabulary head) otherwise."""
    n = _log_int(rng, low, high)
    return n if rng.random() < 0.25 else max(low, n // 64 * 64)


def _multiple(rng, step, low, high):
    return max(low, _log_int(rng, low, high) // step * step)


def _draw_w8a16(rng):
    K, N = _multiple(rng, 128, 1024, 8192), _width(rng, 1000, 14336)
    return {"family": "w8a16", "M": _rows(rng, 2048, 2 * K * N, 1.8e11), "K": K, "N": N,
            "prepared": rng.random() < 0.5}


def _draw_w4a16(rng):
    K, N = _multiple(rng, 128, 1024, 14336), _width(rng, 1000, 14336)
    return {"family": "w4a16", "M": _rows(rng, 4096, 2 * K * N, 1.8e11), "K": K, "N": N,
            "group": rng.choice((64, 128, 128)), "prepared": rng.random() < 0.5}


def _draw_w8a8(rng):
    K, N = _multiple(rng, 128, 1024, 8192), _width(rng, 1000, 14336)
    return {"family": "w8a8", "M": _rows(rng, 4096, 2 * K * N, 5.4e11), "K": K, "N": N}


def _draw_moe(rng, family):
    E = rng.choice((8, 8, 16, 32))
    H = rng.choice((2048, 4096))
    F = _multiple(rng, 128, 1024, 8 * 4096 * 14336 // (E * H) if E * H > 8 * 4096 else 14336)
    top_k = rng.choice((2, 2, 4)) if E > 8 else 2
    T = _rows(rng, 1024, 6 * H * F * top_k, 3.5e11)
    if family == "moe_f16":
        return {"family": family, "T": T, "D": H, "F": F, "E": E, "top_k": top_k}
    return {"family": family, "T": T, "H": H, "F": F, "E": E, "top_k": top_k, "group": 128}


def _draw_fp8_block(rng):
    K, N = _multiple(rng, 128, 1024, 7168), _width(rng, 1000, 14336)
    return {"family": "fp8_block", "M": _rows(rng, 4096, 2 * K * N, 4e11), "K": K, "N": N}


def _draw_q4k(rng):
    return {"family": "q4k", "K": _multiple(rng, 256, 1024, 14336), "N": _width(rng, 1000, 14336)}


def draw(rng):
    family = rng.choice(("w8a16", "w4a16", "w4a16", "w4a16", "w8a8", "w8a8", "moe_w4", "moe_w4", "moe_f16",
                         "fp8_block", "fp8_block", "q4k"))
    if family in ("moe_w4", "moe_f16"):
        return _draw_moe(rng, family)
    return {"w8a16": _draw_w8a16, "w4a16": _draw_w4a16, "w8a8": _draw_w8a8, "fp8_block": _draw_fp8_block,
            "q4k": _draw_q4k}[family](rng)


# ---- inputs ----------------------------------------------------------------------------

def _uniform(g, shape, low, high, dtype):
    return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(low, high, generator=g).to(dtype)


def _normal(g, shape, dtype, std=1.0):
    """N(0, std); large tensors are drawn in parts so that no f32 copy of the whole is needed."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for part in (out if out.dim() == 3 else (out,)):
        part.copy_(torch.randn(part.shape, dtype=torch.float32, device="cuda", generator=g).mul_(std))
    return out


def _bytes(g, shape, low=0, high=256, dtype=torch.uint8):
    return torch.randint(low, high, shape, dtype=dtype, device="cuda", generator=g)


def _w4(g, *lead, K, group):
    return (_bytes(g, (*lead, K // 2)), _uniform(g, (*lead, K // group), 0.005, 0.02, torch.float16),
            _bytes(g, (*lead, K // group), 0, 16))


def _routes(logits, top_k):
    """Ragged expert lists of a token batch: offsets, routes by expert, token and weight of each route."""
    T, E = logits.shape
    top, ids = torch.topk(logits, top_k, dim=1)
    weights = torch.softmax(top, dim=1).reshape(-1).contiguous()
    experts = ids.reshape(-1)
    members = torch.argsort(experts, stable=True).to(torch.int32)
    counts = torch.bincount(experts, minlength=E)
    offsets = torch.zeros(E + 1, dtype=torch.int32, device="cuda")
    offsets[1:] = torch.cumsum(counts, 0)
    tokens = torch.arange(T * top_k, device="cuda", dtype=torch.int32) // top_k
    return offsets, members, tokens, weights


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = case["family"]
    if f == "w8a16":
        return {"x": _normal(g, (case["M"], case["K"]), torch.float16),
                "w": _bytes(g, (case["N"], case["K"]), -127, 128, torch.int8),
                "s": _uniform(g, (case["N"],), 0.002, 0.02, torch.float16)}
    if f == "w4a16":
        q, s, z = _w4(g, case["N"], K=case["K"], group=case["group"])
        return {"x": _normal(g, (case["M"], case["K"]), torch.float16), "q": q, "s": s, "z": z}
    if f == "w8a8":
        return {"x": _normal(g, (case["M"], case["K"]), torch.float16),
                "w": _bytes(g, (case["N"], case["K"]), -127, 128, torch.int8),
                "sw": _uniform(g, (case["N"],), 0.001, 0.01, torch.float32)}
    if f == "moe_w4":
        T, H, F, E = case["T"], case["H"], case["F"], case["E"]
        up, down = _w4(g, E, 2 * F, K=H, group=case["group"]), _w4(g, E, H, K=F, group=case["group"])
        return {"logits": _normal(g, (T, E), torch.float32), "x": _normal(g, (T, H), torch.float16), "up": up,
                "down": down, "residual": _normal(g, (T, H), torch.float32)}
    if f == "moe_f16":
        T, D, F, E = case["T"], case["D"], case["F"], case["E"]
        return {"x": _normal(g, (T, D), torch.float16), "routes": _routes(_normal(g, (T, E), torch.float32), case["top_k"]),
                "w1": _normal(g, (E, D, F), torch.float16, D ** -0.5), "w2": _normal(g, (E, F, D), torch.float16, F ** -0.5),
                "residual": _normal(g, (T, D), torch.float32)}
    if f == "fp8_block":
        M, K, N = case["M"], case["K"], case["N"]
        kb, nb = K // 128, -(-N // 128)
        return {"x": _normal(g, (M, K), torch.bfloat16),
                "w": _normal(g, (N, K), torch.float32).mul_(100.0).clamp_(-448, 448).to(torch.float8_e4m3fn).view(N, kb, 128),
                "sw": _uniform(g, (nb, kb), 1e-4, 4e-4, torch.float32)}
    K, N = case["K"], case["N"]
    w = _bytes(g, (N, K // 256, 144))
    w[..., 0:4] = _uniform(g, (N, K // 256, 2), 0.0005, 0.005, torch.float16).view(torch.uint8)
    return {"w": w, "x": _normal(g, (K // 256, 256), torch.float32)}


def prepare(case, seed):
    state = dict(_inputs(case, seed), case=case)
    f = case["family"]
    if f == "w8a16":
        state["op"] = _artifact(intent.weight_only_int8_matmul)
        state["args"] = (state["x"], state["w"], state["s"])
    elif f == "w4a16":
        state["op"] = _artifact(intent.weight_only_int4_asym_matmul)
        state["args"] = (state["x"], state["q"], state["s"], state["z"])
    elif f == "w8a8":
        state["quantize"] = _artifact(intent.per_token_int8_quantize)
        state["op"] = _artifact(intent.w8a8_scaled_matmul)
    elif f == "moe_w4":
        state["op"] = _artifact(intent.moe_expert_ffn_w4, TOP_K=case["top_k"])
    elif f == "moe_f16":
        state["op"] = _artifact(intent.moe_expert_ffn)
    elif f == "fp8_block":
        state["quantize"] = _artifact(intent.bf16_groupwise_fp8_quantize)
        state["op"] = _artifact(intent.deepgemm_fp8_2xacc)
        state["sx"] = torch.empty(case["M"], case["K"] // 128, dtype=torch.float32, device="cuda")
    else:
        state["op"] = _artifact(intent.quantized_projection)
        state["args"] = (state["w"], state["x"])
    if case.get("prepared"):
        state["bound"] = state["op"].prepare(*state["args"])
    return state


def run(state):
    f = state["case"]["family"]
    if "bound" in state:  # bound once to its buffers, launched per token
        state["bound"].launch()
        return state["bound"].result()
    if f == "w8a8":
        q, sx = state["quantize"].run(state["x"])
        return state["op"].run(q, sx, state["w"], state["sw"])
    if f == "moe_w4":  # the layer adds to the residual stream
        y = state["residual"].clone()
        state["op"](state["logits"], state["x"], *state["up"], *state["down"], y)
        return y
    if f == "moe_f16":
        y = state["residual"].clone()
        state["op"](state["x"], *state["routes"], state["w1"], state["w2"], y)
        return y
    if f == "fp8_block":
        M, K = state["x"].shape
        q = state["quantize"].run(state["x"], state["sx"])
        return state["op"].run(q.view(M, K // 128, 128), state["w"], state["sx"], state["sw"])
    return state["op"].run(*state["args"])


# ---- what a pass cannot do without -------------------------------------------------------

def _experts_used(T, E, top_k):
    """Expected number of experts that a batch of T tokens reaches."""
    return E * (1.0 - (1.0 - top_k / E) ** T)


def work(case):
    f = case["family"]
    if f in ("w8a16", "w8a8"):
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 2 * M * K + N * K + (2 if f == "w8a16" else 4) * N + 2 * M * N, "flops": 2 * M * N * K}
    if f == "w4a16":
        M, K, N, G = case["M"], case["K"], case["N"], case["K"] // case["group"]
        return {"bytes": 2 * M * K + N * K // 2 + 3 * N * G + 2 * M * N, "flops": 2 * M * N * K}
    if f == "moe_w4":
        T, H, F, E, k = case["T"], case["H"], case["F"], case["E"], case["top_k"]
        expert = 3 * H * F // 2 + 3 * (2 * F * (H // case["group"]) + H * (F // case["group"]))
        return {"bytes": int(_experts_used(T, E, k) * expert) + 4 * T * E + 2 * T * H + 8 * T * H,
                "flops": 6 * T * k * H * F}
    if f == "moe_f16":
        T, D, F, E, k = case["T"], case["D"], case["F"], case["E"], case["top_k"]
        return {"bytes": int(_experts_used(T, E, k) * 4 * D * F) + 12 * T * k + 2 * T * D + 8 * T * D,
                "flops": 4 * T * k * D * F}
    if f == "fp8_block":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 2 * M * K + N * K + 4 * (-(-N // 128)) * (K // 128) + 2 * M * N, "flops": 2 * M * N * K}
    K, N = case["K"], case["N"]
    return {"bytes": N * K // 256 * 144 + 4 * K + 4 * N, "flops": 2 * N * K}


def tolerance(case):
    """int8 sums and the K-quant record order are defined bit for bit; the rest round 32-bit sums to 16
    bits, and w4a16 its weights, the experts their hidden values too. Each is four times the distance
    to the 64-bit result: 2.0e-4, 2.9e-4, 4.0e-4 (4.9e-4 for one token), 9.8e-5 and 1.7e-3."""
    f = case["family"]
    if f in ("w8a8", "q4k"):
        return "exact"
    return {"rel": {"w8a16": 8e-4, "w4a16": 1.2e-3, "moe_w4": 1.8e-3, "moe_f16": 4e-4, "fp8_block": 7e-3}[f]}


# ---- 64-bit results ------------------------------------------------------------------------

def _dequant_w4(q, s, z, group):
    w = torch.empty(q.shape[0], q.shape[1] * 2, dtype=torch.float64, device=q.device)
    w[:, 0::2] = (q & 15).double()
    w[:, 1::2] = (q >> 4).double()
    w = w.view(q.shape[0], -1, group)
    w -= z.double().unsqueeze(2)
    w *= s.double().unsqueeze(2)
    return w.view(q.shape[0], -1)


def _exact_moe_w4(case, d):
    logits = d["logits"].double()
    top, ids = torch.topk(logits, case["top_k"], dim=1)
    weights = torch.softmax(top, dim=1)
    y = d["residual"].double()
    for e in range(case["E"]):
        tok, slot = torch.where(ids == e)
        if tok.numel() == 0:
            continue
        gu = d["x"][tok].double() @ _dequant_w4(*(t[e] for t in d["up"]), case["group"]).t()
        gate, up = gu.chunk(2, dim=1)
        out = (torch.nn.functional.silu(gate) * up) @ _dequant_w4(*(t[e] for t in d["down"]), case["group"]).t()
        y.index_add_(0, tok, out * weights[tok, slot].unsqueeze(1))
    return y


def _exact_moe_f16(case, d):
    offsets, members, tokens, weights = d["routes"]
    y = d["residual"].double()
    bounds = offsets.tolist()
    for e in range(case["E"]):
        r = members[bounds[e]:bounds[e + 1]].long()
        if r.numel() == 0:
            continue
        tok = tokens[r].long()
        out = torch.relu(d["x"][tok].double() @ d["w1"][e].double()) @ d["w2"][e].double()
        y.index_add_(0, tok, out * weights[r].double().unsqueeze(1))
    return y


def _exact_fp8_block(case, d):
    M, K, N = case["M"], case["K"], case["N"]
    x = d["x"].float().view(M, K // 128, 128)
    # the quantizer's codes are defined in f32: absmax / 448 (a true quotient), clamp, nearest even
    absmax = x.abs().amax(dim=2, keepdim=True).clamp_min(1e-12)
    scale = absmax / torch.full_like(absmax, 448.0)
    q = (x / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    a = (q.double() * scale.double()).view(M, K)
    rows = torch.arange(N, device="cuda") // 128
    w = (d["w"].double() * d["sw"].double()[rows].unsqueeze(2)).view(N, K)
    return a @ w.t()


def _exact_q4k(case, d):
    w, x = d["w"], d["x"]
    # Q8_K codes are defined in f32: inverse = -127 / extreme (the first of the largest, ties the minimum)
    mx, mn = x.amax(dim=1, keepdim=True), x.amin(dim=1, keepdim=True)
    inverse = torch.full_like(mx, -127.0) / torch.where(mx.abs() > mn.abs(), mx, mn)
    xq = torch.round(x * inverse).clamp(-128, 127).double() * (torch.ones_like(inverse) / inverse).double()
    N, G = w.shape[0], w.shape[1]
    d2 = w[..., 0:4].contiguous().view(torch.float16).double()
    a, b, c = w[..., 4:8], w[..., 8:12], w[..., 12:16]
    sc = torch.cat((a & 63, (c & 15) | ((a >> 6) << 4)), dim=2).double()
    mins = torch.cat((b & 63, (c >> 4) | ((b >> 6) << 4)), dim=2).double()
    nib = w[..., 16:].reshape(N, G, 4, 32)
    vals = torch.stack((nib & 15, nib >> 4), dim=3).reshape(N, G, 8, 32).double()
    full = d2[..., 0, None, None] * sc.unsqueeze(3) * vals - d2[..., 1, None, None] * mins.unsqueeze(3)
    return full.reshape(N, G * 256) @ xq.reshape(-1)


def exact(case, seed):
    d = _inputs(case, seed)
    f = case["family"]
    if f == "w8a16":
        return (d["x"].double() @ d["w"].double().t()) * d["s"].double()
    if f == "w4a16":
        return d["x"].double() @ _dequant_w4(d["q"], d["s"], d["z"], case["group"]).t()
    if f == "w8a8":
        # the quantizer's codes are defined in f32: x * (127 / absmax), clamp, nearest even
        x = d["x"].float()
        absmax = x.abs().amax(dim=1, keepdim=True)
        q = torch.round((x * (torch.full_like(absmax, 127.0) / absmax)).clamp(-128, 127))
        sums = q.double() @ d["w"].double().t()
        return sums * (absmax / torch.full_like(absmax, 127.0)).double() * d["sw"].double()
    if f == "moe_w4":
        return _exact_moe_w4(case, d)
    if f == "moe_f16":
        return _exact_moe_f16(case, d)
    if f == "fp8_block":
        return _exact_fp8_block(case, d)
    return _exact_q4k(case, d)
