"""The work a program has this library do, as cases for timing and for checking outputs.

Every case goes through the package's public entry points (HipOps, LlamaDevice)
with what such a program keeps between calls: device weights in the layouts of
the .cellm formats, a paged f16 K/V cache, prebuilt op lists and output
buffers.  The kinds:

  decode   the four projections of a layer (fused q/k/v rows, o, gate/up rows,
           down), optionally an lm_head, enqueued with one batch call for the
           m sessions decoded together
  prefill  the same layer over the m tokens of a prompt through the fused
           entry points: q/k/v, o, gate/up with its activation, down
  attention  one query row per session (decode), or one per prompt token that
           all read the same pages (prefill), over a paged cache
  step     one whole decode step of the device-resident Llama runner

Weights and scales have the spread of trained ones (normal weights quantized
per row or per group); activations are normal with a few large channels.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cellm_amd import HipOps
from cellm_amd.llama_step import LlamaDevice, LlamaShape

_ops = None


def _hip() -> HipOps:
    """The program's one context."""
    global _ops
    if _ops is None:
        _ops = HipOps(0)
    return _ops


def listed():
    return [
        # Smallest calls: one session of a small int8 model (hidden 576), f32 activations as the
        # norm and embedding ops produce them.  Four launches of a few microseconds.
        dict(name="decode_i8_m1", kind="decode", fmt="i8", xdt="f32", m=1, hidden=576, rows_q=576, rows_kv=192,
             inter=1536, vocab=0),
        # One session of a Qwen2.5-0.5B-shape MLX 4-bit model with its lm_head: bench.py's headline step.
        dict(name="decode_q4_m1_lm_head", kind="decode", fmt="q4", xdt="f16", m=1, hidden=896, rows_q=896,
             rows_kv=128, inter=4864, vocab=151936),
        # Sixteen sessions of a Gemma-3-1B-shape layer decoded together.
        dict(name="decode_q4_m16", kind="decode", fmt="q4", xdt="f16", m=16, hidden=1152, rows_q=1024, rows_kv=256,
             inter=6912, vocab=0),
        # Prompts: 512 tokens of the 4-bit Qwen2.5-0.5B shape with f16 activations (the M=512 qGEMM workload).
        dict(name="prefill_q4_f16_m512", kind="prefill", fmt="q4", xdt="f16", m=512, hidden=896, rows_q=896,
             rows_kv=128, inter=4864, act="silu"),
        # A long prompt through a wide int8 layer (generic 2048 -> 8192 sizes), f16 activations: the largest case.
        dict(name="prefill_i8_f16_m2048", kind="prefill", fmt="i8", xdt="f16", m=2048, hidden=2048, rows_q=2048,
             rows_kv=512, inter=8192, act="silu"),
        # A 512-token prompt of the int8 SmolLM2-360M shape in f32, as a program that chains this library's
        # own f32 ops (embed, RMSNorm, RoPE, attention) has its activations.
        dict(name="prefill_i8_f32_m512", kind="prefill", fmt="i8", xdt="f32", m=512, hidden=960, rows_q=960,
             rows_kv=320, inter=2560, act="silu"),
        # The same for MLX 4-bit weights with f32 scales (what u32 .cellm files hold), a short ragged prompt.
        dict(name="prefill_q4_f32_m200", kind="prefill", fmt="q4", xdt="f32", m=200, hidden=1024, rows_q=1024,
             rows_kv=256, inter=4096, act="silu"),
        # f16 weights (unquantized .cellm tensors), a short ragged prompt, f32 activations.
        dict(name="prefill_f16w_m77", kind="prefill", fmt="f16", xdt="f32", m=77, hidden=896, rows_q=896,
             rows_kv=128, inter=4864, act="silu"),
        # Gemma's MLP format, symmetric 4-bit weights with one scale per row, a 128-token prompt with GELU.
        dict(name="prefill_i4_m128", kind="prefill", fmt="i4", xdt="f32", m=128, hidden=1152, rows_q=1024,
             rows_kv=256, inter=6912, act="gelu"),
        # Eight sessions with long contexts, 32 query heads over 8 kv heads.
        dict(name="attention_decode_8k", kind="attention", prompt=False, rows=8, ctx=8192, n_heads=32, n_kv_heads=8,
             head_dim=128, tokens_per_block=16, window=0),
        # The attention of a 512-token prompt of the Qwen2.5-0.5B shape: every token is a row over the same pages.
        dict(name="attention_prompt_512", kind="attention", prompt=True, rows=512, ctx=512, n_heads=14, n_kv_heads=2,
             head_dim=64, tokens_per_block=16, window=0),
        # A whole decode step with its logits, four sessions near 512 positions: the SmolLM2-360M layer shape
        # and vocabulary, eight layers deep.
        dict(name="step_i8_4_sessions", kind="step", rows=4, n_layers=8, hidden=960, n_heads=15, n_kv_heads=5,
             head_dim=64, inter=2560, vocab=49152, ctx=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "attention", "attention", "step"])
    if kind == "attention":
        head_dim, n_kv, group = rng.choice([64, 128]), rng.randint(1, 8), rng.randint(1, 8)
        prompt = rng.random() < 0.5
        ctx = _log_int(rng, 16, 2048 if prompt else 16384)
        return dict(kind=kind, prompt=prompt, rows=rng.randint(max(1, ctx // 2), ctx) if prompt else rng.randint(1, 16),
                    ctx=ctx, n_heads=n_kv * group, n_kv_heads=n_kv, head_dim=head_dim,
                    tokens_per_block=rng.choice([16, 32]), window=rng.choice([0, 0, 0, 512]))
    if kind == "step":
        head_dim, n_kv, group = 64, rng.randint(1, 5), rng.randint(1, 4)
        return dict(kind=kind, rows=rng.randint(1, 4), n_layers=rng.randint(2, 8), hidden=n_kv * group * head_dim,
                    n_heads=n_kv * group, n_kv_heads=n_kv, head_dim=head_dim, inter=64 * rng.randint(8, 64),
                    vocab=_log_int(rng, 4096, 65536), ctx=_log_int(rng, 16, 2048))
    step = 32 if rng.random() < 0.5 else 64
    hidden = step * (_log_int(rng, 512, 2048) // step)
    rows_kv = 32 * rng.randint(1, 16)
    rows_q = 32 * (_log_int(rng, 512, 2048) // 32)
    inter = step * (_log_int(rng, 1024, 8192) // step)
    if kind == "decode":
        m = _log_int(rng, 1, 64)
        fmt = rng.choice(["i8", "q4", "q4", "i4", "f16", "i2", "q1"])
        if fmt == "q1":  # blocks of 128 along k
            hidden, rows_q, inter = (max(1, v // 128) * 128 for v in (hidden, rows_q, inter))
        xdt = "f32" if m <= 4 and rng.random() < 0.5 or fmt in ("i4", "f16", "i2", "q1") else "f16"
        vocab = _log_int(rng, 16384, 262144) if rng.random() < 0.3 else 0
        return dict(kind=kind, fmt=fmt, xdt=xdt, m=m, hidden=hidden, rows_q=rows_q, rows_kv=rows_kv, inter=inter,
                    vocab=vocab)
    fmt = rng.choice(["i8", "i8", "q4", "q4", "i4", "f16"])
    xdt = rng.choice(["f16", "f32"]) if fmt in ("i8", "q4") else "f32"
    return dict(kind=kind, fmt=fmt, xdt=xdt, m=_log_int(rng, 8, 2048), hidden=hidden, rows_q=rows_q, rows_kv=rows_kv,
                inter=inter, act=rng.choice(["silu", "silu", "gelu"]) if fmt in ("i8", "q4") else
                ("gelu" if fmt == "i4" else "silu"))


# ---- inputs ---------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _x(g, m, k, xdt):
    """Normalised activations with a few large channels."""
    x = torch.randn(m, k, generator=g, device="cuda")
    loud = torch.rand(k, generator=g, device="cuda") < 0.01
    x = x * torch.where(loud, 12.0, 1.0)
    return x.to(torch.float16 if xdt == "f16" else torch.float32)


def _weight(g, fmt, n, k, xdt):
    """One [n, k] weight in a .cellm format: a dict of device tensors."""
    sd = 1.0 / math.sqrt(k)
    if fmt == "f16":
        return dict(w=(torch.randn(n, k, generator=g, device="cuda") * sd).half())
    if fmt == "i8":
        w = (torch.randn(n, k, generator=g, device="cuda") * 32).round_().clamp_(-127, 127).to(torch.int8)
        s = (sd / 32) * (0.5 + torch.rand(n, generator=g, device="cuda"))
        return dict(w=w, s=s.half() if xdt == "f32" else s)
    if fmt == "q4":
        w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
        s = (sd / 4.6) * (0.5 + torch.rand(n, (k + 63) // 64, generator=g, device="cuda"))
        b = -7.5 * s * (0.9 + 0.2 * torch.rand(s.shape, generator=g, device="cuda"))
        # f16 scales beside f16 activations, the f32 scales of u32 .cellm files beside f32 ones
        return dict(w=w, s=s.half(), b=b.half()) if xdt == "f16" else dict(w=w, s=s, b=b)
    if fmt == "i4":
        w = torch.randint(0, 256, (n, (k + 1) // 2), generator=g, device="cuda", dtype=torch.uint8)
        return dict(w=w, s=((sd / 4.6) * (0.5 + torch.rand(n, generator=g, device="cuda"))).half())
    if fmt == "i2":
        w = torch.randint(0, 256, (n, (k + 3) // 4), generator=g, device="cuda", dtype=torch.uint8)
        return dict(w=w, s=(sd * (0.5 + torch.rand(n, generator=g, device="cuda"))).half())
    w = torch.randint(0, 256, (n, k // 128, 18), generator=g, device="cuda", dtype=torch.uint8)  # q1_0_g128
    d = (sd * (0.5 + torch.rand(n, k // 128, generator=g, device="cuda"))).half()
    w[:, :, :2] = d.view(torch.uint8).view(n, k // 128, 2)
    return dict(w=w.view(n, k // 128 * 18))


def _shapes(case):
    """name -> (n, k) of the case's projections."""
    h, q, kv, i = case["hidden"], case["rows_q"], case["rows_kv"], case["inter"]
    if case["kind"] == "decode":
        s = {"qkv": (q + 2 * kv, h), "o": (h, q), "gate_up": (2 * i, h), "down": (h, i)}
        if case["vocab"]:
            s["lm_head"] = (case["vocab"], h)
        return s
    return {"q": (q, h), "k": (kv, h), "v": (kv, h), "o": (h, q), "gate": (i, h), "up": (i, h), "down": (h, i)}


def _projections(case, seed):
    """The weights by name and the activations by their width's role."""
    g = _gen(seed)
    weights = {p: _weight(g, case["fmt"], n, k, case["xdt"]) for p, (n, k) in _shapes(case).items()}
    x = {"x": _x(g, case["m"], case["hidden"], case["xdt"]), "attn": _x(g, case["m"], case["rows_q"], case["xdt"]),
         "h": _x(g, case["m"], case["inter"], case["xdt"])}
    return weights, x


def _input_of(p):
    return {"o": "attn", "down": "h"}.get(p, "x")


def _op(case, w, x, y, k):
    fmt = case["fmt"]
    if fmt == "i8":
        return HipOps.qgemv_op_i8(w["w"], w["s"], x, y)
    if fmt == "q4":
        return HipOps.qgemv_op_q4_affine(w["w"], w["s"], w["b"], x, y)
    if fmt == "i4":
        return HipOps.qgemv_op_i4_sym(w["w"], w["s"], k, x, y, k)
    if fmt == "f16":
        return HipOps.qgemv_op_f16(w["w"], x, y)
    if fmt == "i2":
        return HipOps.qgemv_op_i2(w["w"], w["s"], 0, x, y, k)
    return HipOps.qgemv_op_q1_0_g128(w["w"], x, y, k)


def _prepare_decode(case, seed):
    weights, x = _projections(case, seed)
    shapes = _shapes(case)
    y = {p: torch.empty(case["m"], n, device="cuda") for p, (n, _) in shapes.items()}
    ops = [_op(case, weights[p], x[_input_of(p)], y[p], k) for p, (_, k) in shapes.items()]
    from cellm_amd._lib import QgemvOp

    return dict(kind="decode", ops=(QgemvOp * len(ops))(*ops), y=y, keep=(weights, x))


def _prepare_prefill(case, seed):
    weights, x = _projections(case, seed)
    y = {p: torch.empty(case["m"], n, device="cuda") for p, (n, _) in _shapes(case).items() if p not in ("gate", "up")}
    y["h"] = torch.empty(case["m"], case["inter"], device="cuda")
    state = dict(kind="prefill", case=case, w=weights, x=x, y=y)
    if case["fmt"] == "f16":  # no fused f16 entry point: the up rows need a buffer of their own
        state["up"] = torch.empty(case["m"], case["inter"], device="cuda")
    return state


def _run_prefill(st):
    ops, case, w, x, y = _hip(), st["case"], st["w"], st["x"], st["y"]
    fmt, f16x = case["fmt"], case["xdt"] == "f16"
    if fmt == "i8":
        ops.encode_qkv_i8(w["q"]["w"], w["q"]["s"], w["k"]["w"], w["k"]["s"], w["v"]["w"], w["v"]["s"], x["x"], y["q"],
                          y["k"], y["v"])
        proj = ops.encode_qgemm_i8 if f16x and case["m"] > 64 and case["hidden"] % 64 == 0 == case["rows_q"] % 64 and \
            case["inter"] % 64 == 0 else ops.encode_qgemv_i8
        proj(w["o"]["w"], w["o"]["s"], x["attn"], y["o"])
        gate_up = ops.encode_gate_up_silu_i8 if case["act"] == "silu" else ops.encode_gate_up_gelu_i8
        gate_up(w["gate"]["w"], w["gate"]["s"], w["up"]["w"], w["up"]["s"], x["x"], y["h"])
        proj(w["down"]["w"], w["down"]["s"], x["h"], y["down"])
    elif fmt == "q4":
        q, k, v, g, u = (w[p] for p in ("q", "k", "v", "gate", "up"))
        ops.encode_qkv_q4_affine(q["w"], q["s"], q["b"], k["w"], k["s"], k["b"], v["w"], v["s"], v["b"], x["x"], y["q"],
                                 y["k"], y["v"])
        proj = ops.encode_qgemm_q4_affine if f16x and case["m"] > 64 and case["hidden"] % 64 == 0 == \
            case["rows_q"] % 64 and case["inter"] % 64 == 0 else ops.encode_qgemv_q4_affine
        proj(w["o"]["w"], w["o"]["s"], w["o"]["b"], x["attn"], y["o"])
        gate_up = ops.encode_gate_up_silu_q4_affine if case["act"] == "silu" else ops.encode_gate_up_gelu_q4_affine
        gate_up(g["w"], g["s"], g["b"], u["w"], u["s"], u["b"], x["x"], y["h"])
        proj(w["down"]["w"], w["down"]["s"], w["down"]["b"], x["h"], y["down"])
    elif fmt == "i4":
        h, q, i = case["hidden"], case["rows_q"], case["inter"]
        for p in ("q", "k", "v"):
            ops.encode_qgemv_i4_sym(w[p]["w"], w[p]["s"], h, x["x"], y[p], h)
        ops.encode_qgemv_i4_sym(w["o"]["w"], w["o"]["s"], q, x["attn"], y["o"], q)
        ops.encode_gate_up_gelu_i4_sym(w["gate"]["w"], w["gate"]["s"], w["up"]["w"], w["up"]["s"], h, x["x"], y["h"], h)
        ops.encode_qgemv_i4_sym(w["down"]["w"], w["down"]["s"], i, x["h"], y["down"], i)
    else:
        for p in ("q", "k", "v"):
            ops.encode_qgemv_f16(w[p]["w"], x["x"], y[p])
        ops.encode_qgemv_f16(w["o"]["w"], x["attn"], y["o"])
        ops.encode_qgemv_f16(w["gate"]["w"], x["x"], y["h"])
        ops.encode_qgemv_f16(w["up"]["w"], x["x"], st["up"])
        ops.encode_silu_mul(y["h"], st["up"])
        ops.encode_qgemv_f16(w["down"]["w"], x["h"], y["down"])
    return y


_N_LAYERS, _LAYER = 2, 1  # the attention cases' cache holds two layers, the second is read


def _prepare_attention(case, seed):
    g = _gen(seed)
    rows, ctx, tpb, hd = case["rows"], case["ctx"], case["tokens_per_block"], case["head_dim"]
    per = -(-ctx // tpb)  # blocks of one session
    sessions = 1 if case["prompt"] else rows
    total = per * sessions
    kv_dim = case["n_kv_heads"] * hd
    k, v = (torch.randn(total * _N_LAYERS * tpb * kv_dim, generator=g, device="cuda").half() for _ in range(2))
    tables = torch.randperm(total, generator=g, device="cuda").to(torch.int32).view(sessions, per)
    if case["prompt"]:  # the last `rows` positions of one session
        tables = tables.expand(rows, per).contiguous()
        pos = torch.arange(ctx - rows, ctx, device="cuda", dtype=torch.int32)
    else:  # contexts between half full and full
        pos = torch.randint((ctx - 1) // 2, ctx, (rows,), generator=g, device="cuda", dtype=torch.int32)
    q = torch.randn(rows, case["n_heads"] * hd, generator=g, device="cuda") * 1.5
    return dict(kind="attention", case=case, q=q, k=k, v=v, tables=tables, pos=pos, out=torch.empty_like(q),
                total=total)


def _run_attention(st):
    c = st["case"]
    _hip().encode_attention(st["q"], st["k"], st["v"], st["tables"], st["pos"], st["out"], c["n_heads"],
                            c["n_kv_heads"], c["head_dim"], st["total"], _N_LAYERS, c["tokens_per_block"], _LAYER,
                            window=c["window"])
    return st["out"]


def _step_model(case, seed):
    """The step's host arrays, made on the GPU from the seed."""
    g = _gen(seed)
    shape = LlamaShape(case["n_layers"], case["hidden"], case["n_heads"], case["n_kv_heads"], case["head_dim"],
                       case["inter"], case["vocab"], tokens_per_block=16,
                       total_blocks=case["rows"] * -(-case["ctx"] // 16))

    def norm(n):
        return (1 + 0.1 * torch.randn(n, generator=g, device="cuda")).half().cpu().numpy().view(np.uint16)

    def i8(n, k):
        w = _weight(g, "i8", n, k, "f32")
        return w["w"].cpu().numpy(), w["s"].cpu().numpy().view(np.uint16)

    layers = []
    for _ in range(case["n_layers"]):
        ws = [i8(n, k) for n, k in shape.proj_shapes()]
        layers.append(([w for w, _ in ws], [s for _, s in ws], norm(case["hidden"]), norm(case["hidden"])))
    embed, scale = i8(case["vocab"], case["hidden"])
    kv = [torch.randn(shape.kv_elems(), generator=g, device="cuda").half().cpu().numpy() for _ in range(2)]
    per = shape.total_blocks // case["rows"]
    bt = torch.randperm(shape.total_blocks, generator=g, device="cuda").cpu().numpy().astype(np.uint32)
    pos = torch.randint((case["ctx"] - 1) // 2, case["ctx"], (case["rows"],), generator=g, device="cuda")
    tok = torch.randint(0, case["vocab"], (case["rows"],), generator=g, device="cuda")
    return (shape, layers, embed, scale, norm(case["hidden"]), kv, bt.reshape(case["rows"], per),
            pos.cpu().numpy().astype(np.int32), tok.cpu().numpy().astype(np.uint32))


def _prepare_step(case, seed):
    shape, layers, embed, scale, fnorm, kv, bt, pos, tok = _step_model(case, seed)
    dev = LlamaDevice(shape, layers, embed, scale, fnorm, 0, max_rows=case["rows"], max_blocks=bt.shape[1])
    dev.kv_upload(kv[0], kv[1])
    return dict(kind="step", dev=dev, tok=tok, pos=pos, bt=bt)


def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "attention": _prepare_attention,
            "step": _prepare_step}[case["kind"]](case, seed)


def run(state):
    kind = state["kind"]
    if kind == "decode":
        _hip().encode_qgemv_batch(state["ops"])
        return state["y"]
    if kind == "prefill":
        return _run_prefill(state)
    if kind == "attention":
        return _run_attention(state)
    _, values, logits = state["dev"].step(state["tok"], state["pos"], state["bt"], want_logits=True)
    return dict(values=values, logits=logits)


# ---- what a pass cannot do without --------------------------------------------------


def _weight_bytes(fmt, xdt, n, k):
    groups = (k + 63) // 64
    return {"f16": 2 * n * k, "i8": n * k + (2 if xdt == "f32" else 4) * n,
            "q4": n * k // 2 + n * groups * (4 if xdt == "f16" else 8), "i4": n * ((k + 1) // 2) + 2 * n,
            "i2": n * ((k + 3) // 4) + 2 * n, "q1": n * (k // 128) * 18}[fmt]


def work(case):
    if case["kind"] in ("decode", "prefill"):
        m, xs = case["m"], 2 if case["xdt"] == "f16" else 4
        shapes = _shapes(case)
        nbytes = sum(_weight_bytes(case["fmt"], case["xdt"], n, k) for n, k in shapes.values())
        nbytes += xs * m * (case["hidden"] + case["rows_q"] + case["inter"])
        outs = sum(n for n, _ in shapes.values()) - (case["inter"] if case["kind"] == "prefill" else 0)
        return dict(bytes=nbytes + 4 * m * outs, flops=2 * m * sum(n * k for n, k in shapes.values()))
    if case["kind"] == "attention":
        rows, ctx, hd = case["rows"], case["ctx"], case["head_dim"]
        # decode contexts are spread over half full to full
        lens = [p + 1 for p in range(ctx - rows, ctx)] if case["prompt"] else [0.75 * ctx] * rows
        seen = [min(n, case["window"]) if case["window"] else n for n in lens]
        if case["prompt"]:
            read = min(ctx, case["window"] + rows - 1) if case["window"] else ctx
        else:
            read = sum(seen)
        return dict(bytes=4 * case["n_kv_heads"] * hd * read + 8 * rows * case["n_heads"] * hd,
                    flops=4 * hd * case["n_heads"] * sum(seen))
    h, kv, i = case["hidden"], case["n_kv_heads"] * case["head_dim"], case["inter"]
    per_layer = 2 * h * h + 2 * kv * h + 3 * i * h
    lens = 0.75 * case["ctx"] * case["rows"]
    return dict(bytes=case["n_layers"] * (per_layer + 4 * kv * lens) + case["vocab"] * (h + 2 + 4 * case["rows"]),
                flops=2 * case["rows"] * (case["n_layers"] * per_layer + case["vocab"] * h) +
                4 * case["n_layers"] * h * lens)


def tolerance(case):
    """About four times the error measured against 64-bit results."""
    if case["kind"] == "step":  # sums reordered in one layer travel through the others (and K/V rounds to f16)
        return {"rel": 5e-5}
    if case["kind"] == "attention":
        return {"rel": 2e-6}
    if case["fmt"] == "q4" and case["xdt"] == "f16":
        # from 2 rows on 4-bit affine weights meet f16 activations as f16 weights (2^-11 each)
        return {"rel": 1e-3 if case["m"] > 1 else 4e-5}
    if case["kind"] == "decode" and case["vocab"] and case["xdt"] == "f32":
        # long f32 outputs may hold activations as integers of 2^-20 of their row's largest
        return {"rel": 5e-5}
    return {"rel": 3e-6}  # exact products of exact weights, 32-bit sums


# ---- 64-bit results -----------------------------------------------------------------


def _dequant64(fmt, w, k):
    if fmt == "f16":
        return w["w"].double()
    if fmt == "i8":
        return w["w"].double() * w["s"].double()[:, None]
    if fmt == "q4":
        sh = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
        q = ((w["w"][:, :, None] >> sh) & 15).reshape(w["w"].shape[0], k).double()
        s, b = (w[p].double().repeat_interleave(64, 1)[:, :k] for p in ("s", "b"))
        return q * s + b
    if fmt == "i4":
        q = torch.stack([w["w"] & 15, w["w"] >> 4], 2).reshape(w["w"].shape[0], -1)[:, :k]
        return (q.double() - 8) * w["s"].double()[:, None]
    if fmt == "i2":
        q = torch.stack([(w["w"] >> (2 * j)) & 3 for j in range(4)], 2).reshape(w["w"].shape[0], -1)[:, :k]
        return (q.double() - 1.5) * w["s"].double()[:, None]
    blocks = w["w"].view(w["w"].shape[0], k // 128, 18)
    d = blocks[:, :, :2].contiguous().view(torch.float16).double()
    bits = torch.stack([(blocks[:, :, 2:] >> j) & 1 for j in range(8)], 3).reshape(w["w"].shape[0], k // 128, 128)
    return ((bits.double() * 2 - 1) * d).reshape(-1, k)


def _gelu_tanh(g):
    return 0.5 * g * (1 + torch.tanh(0.7978846 * (g + 0.044715 * g * g * g)))


def _exact_projections(case, seed):
    weights, x = _projections(case, seed)
    y = {}
    for p, (_, k) in _shapes(case).items():
        y[p] = torch.matmul(x[_input_of(p)].double(), _dequant64(case["fmt"], weights[p], k).t().contiguous())
    if case["kind"] == "prefill":
        g = y.pop("gate")
        y["h"] = (g / (1 + torch.exp(-g)) if case["act"] == "silu" else _gelu_tanh(g)) * y.pop("up")
    return y


def _kv64(k, v, table, length, layer, n_layers, tpb, n_kv, hd):
    """K and V [n_kv, length, hd] of one session's first `length` positions."""
    pages = [a.view(-1, n_layers, tpb, n_kv, hd)[table.long(), layer].reshape(-1, n_kv, hd)[:length] for a in (k, v)]
    return [a.double().transpose(0, 1).contiguous() for a in pages]


def _attend64(q, k, v, lens, window):
    """q [rows, n_heads, hd] over k, v [n_kv, length, hd]; row r sees positions lens[r] - window .. lens[r] - 1."""
    rows, nh, hd = q.shape
    n_kv = k.shape[0]
    t = torch.arange(k.shape[1], device=k.device)
    first = (lens - window).clamp(min=0) if window else torch.zeros_like(lens)
    hidden = (t[None] >= lens[:, None]) | (t[None] < first[:, None])
    out = torch.empty_like(q)
    for h in range(nh):
        kv = h // (nh // n_kv)
        s = torch.matmul(q[:, h].contiguous(), k[kv].t().contiguous()) / math.sqrt(hd)
        out[:, h] = torch.matmul(torch.softmax(s.masked_fill(hidden, -math.inf), 1), v[kv])
    return out.reshape(rows, nh * hd)


def _exact_attention(case, seed):
    st = _prepare_attention(case, seed)
    q = st["q"].double().view(case["rows"], case["n_heads"], case["head_dim"])
    lens = st["pos"].long() + 1

    def attend(rows):
        k, v = _kv64(st["k"], st["v"], st["tables"][rows.start], int(lens[rows].max()), _LAYER, _N_LAYERS,
                     case["tokens_per_block"], case["n_kv_heads"], case["head_dim"])
        return _attend64(q[rows], k, v, lens[rows], case["window"])

    if case["prompt"]:
        return attend(slice(0, case["rows"]))
    return torch.cat([attend(slice(r, r + 1)) for r in range(case["rows"])])


def _exact_step(case, seed):
    shape, layers, embed, scale, fnorm, kv, bt, pos, tok = _step_model(case, seed)

    def f16(bits):
        return torch.from_numpy(np.ascontiguousarray(bits).view(np.float16)).cuda().double()

    def i8(w, s):
        return torch.from_numpy(w).cuda().double() * f16(s)[:, None]

    def norm(v, w):
        return v / torch.sqrt((v * v).mean(1, keepdim=True) + shape.rms_norm_eps) * f16(w)

    def mul(v, w, s):
        return torch.matmul(v, i8(w, s).t().contiguous())

    rows, nh, nkv, hd = case["rows"], case["n_heads"], case["n_kv_heads"], case["head_dim"]
    p = torch.from_numpy(pos).cuda().long()
    ang = p.double()[:, None] * shape.rope_theta ** (-torch.arange(hd // 2, device="cuda").double() * 2 / hd)
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def rope(v, heads):
        a, b = v.view(rows, heads, hd).chunk(2, 2)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], 2)

    kc, vc = (torch.from_numpy(a).cuda() for a in kv)
    table = torch.from_numpy(bt.astype(np.int64)).cuda()
    where = table.gather(1, (p // 16)[:, None])[:, 0]
    emb = i8(embed, scale)
    x = emb[torch.from_numpy(tok.astype(np.int64)).cuda()]
    for layer, (ws, ss, n1, n2) in enumerate(layers):
        xn = norm(x, n1)
        q = rope(mul(xn, ws[0], ss[0]), nh)
        for cache, new in ((kc, rope(mul(xn, ws[1], ss[1]), nkv)), (vc, mul(xn, ws[2], ss[2]).view(rows, nkv, hd))):
            cache.view(-1, shape.n_layers, 16, nkv, hd)[where, layer, p % 16] = new.half()
        att = []
        for r in range(rows):
            k, v = _kv64(kc, vc, table[r], int(pos[r]) + 1, layer, shape.n_layers, 16, nkv, hd)
            att.append(_attend64(q[r:r + 1], k, v, p[r:r + 1] + 1, 0))
        x = x + mul(torch.cat(att), ws[3], ss[3])
        xn = norm(x, n2)
        g = mul(xn, ws[4], ss[4])
        x = x + mul(g / (1 + torch.exp(-g)) * mul(xn, ws[5], ss[5]), ws[6], ss[6])
    logits = torch.matmul(norm(x, fnorm), emb.t().contiguous())
    return dict(values=logits.max(1).values, logits=logits)


def exact(case, seed):
    if case["kind"] == "attention":
        return _exact_attention(case, seed)
    if case["kind"] == "step":
        return _exact_step(case, seed)
    return _exact_projections(case, seed)
