"""The work this framework's users have it do, as measurable cases.

Every case calls the public entry points a program with its activations in
HBM calls: device.linear and device.ffn (the quantized projections), and the
C ABI through _ffi for the routed experts (rk_npu_hip_moe_run) and for the
attention layer (truncate to the position, append the step's K/V rows, run).
Weights, workspaces, caches and output buffers are what such a program keeps;
one pass is one layer call on the caller's stream.

Sizes: hidden 2560, FFN 9728, 32 query and 8 KV heads of 128 (the dense
model of the benchmark), hidden 2048 with 128 experts, top 8 and intermediate
768 (its MoE), head_dim 64 / 128 / 256 (the attention kernels' range), batches
of 1 and 4 (decode), 16 (a draft verification or batched decode), 64 and 128
(the reference's micro-batches), 512 and 4096 (whole prompts), 25 tokens (a
short MoE chunk), and ragged sizes among the drawn cases.

Activations are normal with 0.5% of the channels 20 times larger, rounded to
fp16; weight codes are uniform, column scales uniform in 0.001..0.01.
"""
from __future__ import annotations

import ctypes
import math

import torch

from open_rknpu2_lm_infer_amd import _ffi as F
from open_rknpu2_lm_infer_amd import device as D
from open_rknpu2_lm_infer_amd import npu

H, FF = 2560, 9728


# --- the cases ---------------------------------------------------------------

def listed():
    return [
        # one decode step's fused q/k/v projection: latency of a single launch
        linear("decode_qkv_w4", 1, H, 6144, 4, "f16"),
        # one decode step's FFN: gate/up, SwiGLU, requantization, down
        ffn("decode_ffn_w4", 1, H, FF, 4, 4, "f16"),
        # one decode step of a routed layer
        moe("decode_moe", 1, 2048, 768, 128, 8, 8),
        # one decode step's attention over a filled context
        attention("decode_attention", 1, 3967, 32, 8, 128, True, "f16"),
        # several sequences' (or a draft's) tokens through the o projection
        linear("verify_o_w4_m16", 16, 4096, H, 4, "f16"),
        # a micro-batch of 64 tokens through the FFN, f32 activations
        ffn("chunk_ffn_w4_m64", 64, H, FF, 4, 4, "f32"),
        # the reference's 128-token micro-batch, W8 up projection
        linear("chunk_up_w8_m128", 128, H, FF, 8, "f16"),
        # a short chunk through a routed layer: few tokens per expert
        moe("chunk_moe_t25", 25, 2048, 768, 128, 8, 8),
        # a 512-token prompt through a routed layer
        moe("prompt_moe_t512", 512, 2048, 768, 128, 8, 8),
        # a micro-batch of queries at the end of a filled context
        attention("chunk_attention_d128", 128, 3968, 32, 8, 128, True, "f16"),
        # the same with wide heads (few KV heads of 256)
        attention("chunk_attention_d256", 128, 1920, 16, 2, 256, True, "f32"),
        # a whole prompt through the FFN: the largest call
        ffn("prompt_ffn_m4096", 4096, H, FF, 4, 8, "f16"),
    ]


def linear(name, rows, k, n, bits, dtype, swiglu=False):
    return {"name": name, "kind": "linear", "rows": rows, "k": k, "n": n, "bits": bits, "dtype": dtype,
            "swiglu": swiglu}


def ffn(name, rows, h, f, gu_bits, dn_bits, dtype):
    return {"name": name, "kind": "ffn", "rows": rows, "h": h, "f": f, "gu_bits": gu_bits, "dn_bits": dn_bits,
            "dtype": dtype}


def moe(name, rows, h, inter, experts, top, dn_bits):
    return {"name": name, "kind": "moe", "rows": rows, "h": h, "inter": inter, "experts": experts, "top": top,
            "dn_bits": dn_bits}


def attention(name, rows, position, qh, kh, d, causal, dtype):
    return {"name": name, "kind": "attention", "rows": rows, "position": position, "qh": qh, "kh": kh, "d": d,
            "causal": causal, "dtype": dtype}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A dimension: mostly a multiple of 64, sometimes of 16, sometimes any."""
    v = _log(rng, lo, hi)
    step = rng.choice([64, 64, 64, 16, 1])
    return max(lo, v // step * step)


def draw(rng):
    kind = rng.choice(["linear", "linear", "ffn", "moe", "attention", "attention"])
    if kind == "linear":
        bits = rng.choice([4, 8])
        swiglu = rng.random() < 0.25
        k, n = _size(rng, 512, FF), _size(rng, 512, 2 * FF)
        if swiglu:
            n = max(64, n // 64 * 64)
        case = linear("", _log(rng, 1, 4096), k, n, bits, rng.choice(["f16", "f32"]), swiglu)
    elif kind == "ffn":
        case = ffn("", _log(rng, 1, 2048), _size(rng, 512, 4096), max(512, _log(rng, 1024, FF) // 32 * 32),
                   rng.choice([4, 4, 8]), rng.choice([4, 8]), rng.choice(["f16", "f32"]))
    elif kind == "moe":
        case = moe("", _log(rng, 1, 512), rng.choice([1024, 1536, 2048]), _log(rng, 256, 768) // 32 * 32,
                   rng.choice([32, 64, 128]), rng.choice([2, 4, 8]), rng.choice([4, 8]))
    else:
        kh = rng.choice([1, 2, 4, 8])
        d = rng.choice([64, 128, 256])
        rows = _log(rng, 1, 128)
        case = attention("", rows, _log(rng, 64, 16384) - 1, kh * rng.choice([1, 2, 4, 8]), kh, d,
                         rng.random() < 0.75, rng.choice(["f16", "f32"]))
    del case["name"]
    return case


# --- inputs ------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _codes(g, bits, k, n):
    lo, hi = (-8, 8) if bits == 4 else (-127, 128)
    return torch.randint(lo, hi, (k, n), generator=g, device="cuda", dtype=torch.int8)


def _scales(g, n):
    return torch.rand(n, generator=g, device="cuda") * 0.009 + 0.001


def _rows(g, rows, k):
    x = torch.randn(rows, k, generator=g, device="cuda")
    outlier = torch.randperm(k, generator=g, device="cuda")[:math.ceil(0.005 * k)]
    x[:, outlier] *= 20.0
    return x.half()


def _dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.float32


def _inputs(case, seed):
    """The case's inputs, a function of the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        return {"codes": _codes(g, case["bits"], case["k"], case["n"]), "scales": _scales(g, case["n"]),
                "x": _rows(g, case["rows"], case["k"]).to(_dtype(case))}
    if kind == "ffn":
        h, f = case["h"], case["f"]
        return {"gu": (_codes(g, case["gu_bits"], h, 2 * f), _scales(g, 2 * f)),
                "dn": (_codes(g, case["dn_bits"], f, h), _scales(g, h)),
                "x": _rows(g, case["rows"], h).to(_dtype(case))}
    if kind == "moe":
        h, inter, e, t = case["h"], case["inter"], case["experts"], case["rows"]
        gu = torch.randint(-8, 8, (e, h, 2 * inter), generator=g, device="cuda", dtype=torch.int8)
        lo, hi = (-8, 8) if case["dn_bits"] == 4 else (-127, 128)
        dn = torch.randint(lo, hi, (e, inter, h), generator=g, device="cuda", dtype=torch.int8)
        gus = torch.rand(e, 2 * inter, generator=g, device="cuda") * 0.009 + 0.001
        dns = torch.rand(e, h, generator=g, device="cuda") * 0.009 + 0.001
        logits = torch.randn(t, e, generator=g, device="cuda")
        top = torch.topk(logits, case["top"], dim=1)
        return {"gu": gu, "gus": gus, "dn": dn, "dns": dns, "x": _rows(g, t, h).float(),
                "ids": top.indices.to(torch.int32).contiguous(),
                "routes": torch.softmax(top.values, dim=1).contiguous()}
    rows, length, kh, d = case["rows"], case["position"] + case["rows"], case["kh"], case["d"]
    half = dict(generator=g, device="cuda", dtype=torch.float16)
    return {"q": torch.randn(case["qh"], rows, d, **half), "k": torch.randn(kh, length, d, **half),
            "v": torch.randn(kh, length, d, **half)}


# --- what a program holds, and one pass ----------------------------------------

def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    ctx = D.DeviceContext(0)
    state = {"kind": kind, "ctx": ctx, "rows": case["rows"]}
    if kind == "linear":
        rows, k, n, bits = case["rows"], case["k"], case["n"], case["bits"]
        state.update(w=ctx.weights(bits, x["codes"], x["scales"]), x=x["x"], swiglu=case["swiglu"],
                     out=torch.empty(rows, n // 2 if case["swiglu"] else n, dtype=_dtype(case), device="cuda"),
                     ws=ctx.workspace(bits, rows, k, n))
    elif kind == "ffn":
        rows, h, f = case["rows"], case["h"], case["f"]
        state.update(gu=ctx.weights(case["gu_bits"], *x["gu"]), dn=ctx.weights(case["dn_bits"], *x["dn"]), x=x["x"],
                     out=torch.empty(rows, h, dtype=_dtype(case), device="cuda"),
                     gws=ctx.workspace(case["gu_bits"], rows, h, 2 * f), dws=ctx.workspace(case["dn_bits"], rows, f, h))
    elif kind == "moe":
        state.update(_moe_handles(case, ctx, x), x=x["x"], ids=x["ids"], routes=x["routes"],
                     out=torch.empty_like(x["x"]))
    else:
        state.update(_attention_handles(case, ctx, x))
    torch.cuda.synchronize()
    return state


def _moe_handles(case, ctx, x):
    L = F.lib()
    h, inter, e = case["h"], case["inter"], case["experts"]
    host = {n: x[n].cpu() for n in ("gu", "gus", "dn", "dns")}

    def at(name, ctype, i):
        return ctypes.cast(host[name][i].data_ptr(), ctypes.POINTER(ctype))

    experts = (F.rk_npu_moe_w8_expert * e)()
    for i in range(e):
        experts[i] = F.rk_npu_moe_w8_expert(at("gu", ctypes.c_int8, i), at("gus", ctypes.c_float, i),
                                            at("dn", ctypes.c_int8, i), at("dns", ctypes.c_float, i))
    cfg = F.rk_npu_moe_w8_config()
    L.rk_npu_moe_w8_config_init(ctypes.byref(cfg), h, inter, e, 0, case["top"], case["rows"])
    if case["dn_bits"] == 8:
        create, work = L.rk_npu_moe_w4w8_weights_create, L.rk_npu_moe_w4w8_workspace_create
    else:
        create, work = L.rk_npu_moe_quant_weights_create, L.rk_npu_moe_quant_workspace_create
    return {"bank": npu._Handle(create(ctx.domain, ctypes.byref(cfg.weights), experts), L.rk_npu_moe_w8_weights_free,
                                "MoE bank", ctx.shared),
            "ws": npu._Handle(work(ctx.domain, ctypes.byref(cfg)), L.rk_npu_moe_w8_workspace_free, "MoE workspace",
                              ctx.shared)}


def _attention_handles(case, ctx, x):
    L = F.lib()
    rows, pos = case["rows"], case["position"]
    capacity = -(-(pos + rows) // 32) * 32
    cfg = F.rk_npu_attention_f16_config()
    L.rk_npu_attention_f16_config_init(ctypes.byref(cfg))
    cfg.query_heads, cfg.kv_heads, cfg.head_dim = case["qh"], case["kh"], case["d"]
    cfg.softmax_scale = case["d"] ** -0.5
    cfg.max_query_rows, cfg.max_capacity, cfg.initial_capacity = rows, capacity, capacity
    cfg.mask_mode = F.RK_NPU_ATTENTION_F16_CAUSAL if case["causal"] else F.RK_NPU_ATTENTION_F16_NO_MASK
    ws, cache = ctypes.c_void_p(), ctypes.c_void_p()
    npu.check(L.rk_npu_attention_f16_prepare(ctx.domain, ctypes.byref(cfg), ctypes.byref(ws)), "prepare attention")
    ws = npu._Handle(ws.value, L.rk_npu_attention_f16_workspace_free, "attention workspace", ctx.shared)
    npu.check(L.rk_npu_attention_f16_cache_create(ctx.domain, ctypes.byref(cfg), ctypes.byref(cache)), "KV cache")
    cache = npu._Handle(cache.value, L.rk_npu_attention_f16_cache_free, "KV cache", ctx.shared)
    old = [x[n][:, :pos].contiguous() for n in ("k", "v")]
    new = [x[n][:, pos:].contiguous() for n in ("k", "v")]
    npu.check(L.rk_npu_hip_attention_cache_append(cache.raw, old[0].data_ptr(), old[1].data_ptr(), pos,
                                                  D.current_stream()), "fill the KV cache")
    torch.cuda.synchronize()
    return {"attn": ws, "cache": cache, "q": x["q"], "k": new[0], "v": new[1], "position": pos,
            "f16": case["dtype"] == "f16", "out": torch.empty(x["q"].shape, dtype=_dtype(case), device="cuda")}


def run(state):
    L = F.lib()
    kind, out, rows = state["kind"], state["out"], state["rows"]
    if kind == "linear":
        D.linear(state["ctx"], state["w"], state["x"], out, rows, swiglu=state["swiglu"], ws=state["ws"])
    elif kind == "ffn":
        D.ffn(state["ctx"], state["gu"], state["dn"], state["x"], out, rows, gws=state["gws"], dws=state["dws"])
    elif kind == "moe":
        npu.check(L.rk_npu_hip_moe_run(state["ws"].raw, state["bank"].raw, rows, state["x"].data_ptr(),
                                       state["ids"].data_ptr(), state["routes"].data_ptr(), out.data_ptr(),
                                       D.current_stream()), "device MoE")
    else:
        stream, cache, pos = D.current_stream(), state["cache"].raw, state["position"]
        npu.check(L.rk_npu_attention_f16_cache_truncate(cache, pos), "truncate")
        npu.check(L.rk_npu_hip_attention_cache_append(cache, state["k"].data_ptr(), state["v"].data_ptr(), rows,
                                                      stream), "append")
        npu.check(L.rk_npu_hip_attention_run(state["attn"].raw, cache, state["q"].data_ptr(), rows, pos,
                                             out.data_ptr(), 1 if state["f16"] else 0, stream), "attention")
    return out


# --- what a pass cannot do without --------------------------------------------

def work(case):
    kind, rows = case["kind"], case["rows"]
    esz = 2 if case.get("dtype") == "f16" else 4
    if kind == "linear":
        k, n, bits = case["k"], case["n"], case["bits"]
        out = n // 2 if case["swiglu"] else n
        return {"bytes": k * n * bits // 8 + 4 * n + rows * (k + out) * esz, "flops": 2 * rows * k * n}
    if kind == "ffn":
        h, f = case["h"], case["f"]
        return {"bytes": 2 * h * f * case["gu_bits"] // 8 + 8 * f + h * f * case["dn_bits"] // 8 + 4 * h +
                2 * rows * h * esz, "flops": 6 * rows * h * f}
    if kind == "moe":
        h, inter, e, top = case["h"], case["inter"], case["experts"], case["top"]
        used = e * (1.0 - (1.0 - top / e) ** rows)  # experts that some token of the batch takes
        expert = h * inter + 8 * inter + h * inter * case["dn_bits"] // 8 + 4 * h
        return {"bytes": int(used * expert) + 8 * rows * h + 8 * rows * top, "flops": 6 * rows * top * h * inter}
    qh, kh, d, pos = case["qh"], case["kh"], case["d"], case["position"]
    keys = rows * (pos + (rows + 1) / 2) if case["causal"] else rows * (pos + rows)
    return {"bytes": 4 * kh * (pos + rows) * d + 8 * kh * rows * d + qh * rows * d * (2 + esz),
            "flops": int(4 * qh * d * keys)}


def tolerance(case):
    kind = case["kind"]
    if kind == "attention":
        # fp16 softmax weights (2^-11 each, random signs) and fp16 outputs:
        # 2.9e-4 measured against 64 bits
        return {"rel": 1.2e-3}
    if kind == "linear":
        # exact integer sums, two f32 multiplications; fp16 outputs round once
        # (2.1e-4 measured against 64 bits)
        return {"rel": 1e-3 if case["dtype"] == "f16" else 1e-5}
    # the middle is requantized to 8 bits: a last-bit difference before it
    # moves a code now and then (2.2e-4 measured with fp16 outputs)
    return {"rel": 1e-3}


# --- the same in 64 bits -------------------------------------------------------

def _quantized(x, even):
    """Codes (as float64) and scales of rows: absmax / 127, the scaled value
    rounded half away from zero (dense) or half to even (experts). The codes
    are part of the operation's definition, f32 arithmetic included."""
    x = x.float()
    m = x.abs().amax(dim=1, keepdim=True)
    s = m / 127.0
    if not even:
        s = s.clamp_min(torch.finfo(torch.float32).tiny)
    s = torch.where(m == 0, torch.ones_like(s), s)
    v = x * (1.0 / s)
    q = torch.round(v) if even else torch.trunc(v.double() + torch.copysign(torch.full_like(v, 0.5), v).double())
    return q.double().clamp(-127, 127), s.double()


def _product(x, codes, scales, even=False):
    q, s = _quantized(x, even)
    return (q @ codes.double()) * s * scales.double()


def _swiglu(y):
    g, u = y.chunk(2, dim=1)
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        parts = []
        for r in range(0, case["rows"], 1024):
            y = _product(x["x"][r:r + 1024], x["codes"], x["scales"])
            parts.append(_swiglu(y) if case["swiglu"] else y)
        return torch.cat(parts)
    if kind == "ffn":
        parts = []
        for r in range(0, case["rows"], 1024):
            mid = _swiglu(_product(x["x"][r:r + 1024], *x["gu"]))
            parts.append(_product(mid, *x["dn"]))
        return torch.cat(parts)
    if kind == "moe":
        out = torch.zeros(case["rows"], case["h"], dtype=torch.float64, device="cuda")
        for e in range(case["experts"]):
            tok, rank = torch.nonzero(x["ids"] == e, as_tuple=True)
            if tok.numel() == 0:
                continue
            mid = _swiglu(_product(x["x"][tok], x["gu"][e], x["gus"][e], True))
            y = _product(mid, x["dn"][e], x["dns"][e], True)
            out.index_add_(0, tok, y * x["routes"][tok, rank].double()[:, None])
        return out
    rows, pos, d, group = case["rows"], case["position"], case["d"], case["qh"] // case["kh"]
    out = torch.empty(case["qh"], rows, d, dtype=torch.float64, device="cuda")
    scale = float(torch.tensor(d ** -0.5, dtype=torch.float32))
    keys = torch.arange(pos + rows, device="cuda")
    hidden = keys[None, :] > (pos + torch.arange(rows, device="cuda"))[:, None]
    for h in range(case["qh"]):
        k, v = x["k"][h // group].double(), x["v"][h // group].double()
        s = (x["q"][h].double() @ k.t().contiguous()) * scale
        if case["causal"]:
            s.masked_fill_(hidden, -math.inf)
        out[h] = torch.softmax(s, dim=1) @ v
    return out
