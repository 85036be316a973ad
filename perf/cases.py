"""Performance cases of the quantized-linear path, and how each is run.

A case names a workload a program has this library do: the linear layers of a
decoder (decode, batched decode, prefill) over packed weights, a routed expert
FFN, or the W8A8 linear.  `prepare` makes what such a program holds (weights,
activations, output buffers, bound calls), `run` is one pass through the
public entry points, `exact` the same result in float64 from plain torch.

Sizes: the Qwen3-8B linear shapes (hidden 4096, q|k|v 6144, gate|up 24576,
down 12288 -> 4096), the Qwen3-30B-A3B-like expert layer (hidden 2048, 128
experts of 768, top-8), the 2048 x 2048 Q8_0 GEMV of the bench_matmul_rlx
harness, and generic ones between them.
"""
from __future__ import annotations

import sys
from pathlib import Path

import torch

_ROOT = Path(__file__).resolve().parent.parent
if str(_ROOT / "rlx-models_amd") not in sys.path:
    sys.path.insert(0, str(_ROOT / "rlx-models_amd"))

import rlxq  # noqa: E402

_SCHEME = {"q8_0": rlxq.GGUF_Q8_0, "q4_1": rlxq.GGUF_Q4_1, "q4_k": rlxq.GGUF_Q4_K, "q6_k": rlxq.GGUF_Q6_K,
           "mlx4": rlxq.MLX_AFFINE4}
_BPW = {"q8_0": 34 / 32, "q4_1": 20 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256, "mlx4": 0.5 + 4 / 64}
_DT = {"f32": torch.float32, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "bf16": 2}
_GROUP = 64   # MLX group size

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = rlxq.Context(0)
    return _ctx


# ---- the cases -------------------------------------------------------------
def _decoder(name, m, scheme, down, x, y, layers, hidden=4096, qkv=6144, inter=12288):
    """The four linear calls of `layers` decoder layers on m rows: q|k|v,
    o, gate|up (of `scheme`) and down (of `down`)."""
    c = {"kind": "decoder", "m": m, "scheme": scheme, "down": down, "x": x, "y": y, "layers": layers,
         "hidden": hidden, "qkv": qkv, "inter": inter}
    return {"name": name, **c} if name else c


def _linear(name, m, k, n, scheme, x, y, layers=1):
    """One linear call, `layers` times over weights of their own."""
    c = {"kind": "linear", "m": m, "k": k, "n": n, "scheme": scheme, "x": x, "y": y, "layers": layers}
    return {"name": name, **c} if name else c


def _moe(name, tokens, scheme, x, experts=128, hidden=2048, inter=768, top_k=8):
    """Router, gate|up + SwiGLU and down + weighted sum of one expert FFN."""
    c = {"kind": "moe", "m": tokens, "scheme": scheme, "x": x, "experts": experts, "hidden": hidden,
         "inter": inter, "top_k": top_k}
    return {"name": name, **c} if name else c


def _w8a8(name, m, k, n):
    c = {"kind": "w8a8", "m": m, "k": k, "n": n}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest calls: the bench_matmul_rlx GEMV, launch latency and little else
        _linear("gemv_q8_0_2048_f32", 1, 2048, 2048, "q8_0", "f32", "f32", 4),
        # single-stream decode, layer after layer (more weights than the caches hold)
        _decoder("decode_q4_1_m1_bf16", 1, "q4_1", "q4_1", "bf16", "f32", 3),
        # the same on a Q4_K_M-like checkpoint with the reference's operand types
        _decoder("decode_q4_k_m_m1_f32", 1, "q4_k", "q6_k", "f32", "f32", 3),
        # four streams (or four drafted tokens) on an MLX 4-bit checkpoint
        _decoder("decode_mlx4_m4_bf16", 4, "mlx4", "mlx4", "bf16", "f32", 3),
        # batched decode, 16 and 64 streams
        _decoder("batch16_q8_0_bf16", 16, "q8_0", "q8_0", "bf16", "f32", 2),
        _decoder("batch64_q4_1_f32", 64, "q4_1", "q4_1", "f32", "f32", 2),
        # a short prompt of an odd length on the Q4_K_M-like checkpoint
        _decoder("prompt197_q4_k_m_f32", 197, "q4_k", "q6_k", "f32", "f32", 1),
        # a prompt chunk with the reference's operand types
        _decoder("prefill512_q4_1_f32", 512, "q4_1", "q4_1", "f32", "f32", 1),
        # long-prompt prefill in bf16: the largest
        _decoder("prefill4096_q4_1_bf16", 4096, "q4_1", "q4_1", "bf16", "bf16", 1),
        # the W8A8 linear at a prefill size (gate|up)
        _w8a8("w8a8_2048_bf16", 2048, 4096, 24576),
        # a routed expert layer: 16 decoding streams, and a 256-token prompt
        _moe("moe16_q4_1_bf16", 16, "q4_1", "bf16"),
        _moe("moe256_q4_k_f32", 256, "q4_k", "f32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """A case of the listed ones' ranges: rows 1 to 4096 over their logarithm,
    the listed formats and operand types, hidden sizes 1024 to 5120."""
    kind = rng.choice(["linear", "decoder", "decoder", "decoder", "decoder", "moe", "moe", "w8a8"])
    if kind == "linear":
        scheme = rng.choice(sorted(_SCHEME))
        # (an output width that is not a multiple of any tile)
        return _linear(None, _log_int(rng, 1, 16), 256 * rng.randint(4, 20), 2 * rng.randint(500, 4000) + 1, scheme,
                       rng.choice(["f32", "bf16"]), "f32")
    if kind == "moe":
        return _moe(None, _log_int(rng, 2, 384), rng.choice(["q4_1", "q4_k"]), rng.choice(["f32", "bf16"]),
                    hidden=256 * rng.randint(5, 9), inter=256 * rng.randint(2, 4))
    if kind == "w8a8":
        return _w8a8(None, _log_int(rng, 64, 3072), 256 * rng.randint(6, 16), 16 * rng.randint(100, 1500))
    scheme = rng.choice(["q4_1", "q4_k", "q4_k", "mlx4", "q8_0"])
    down = rng.choice(["q4_k", "q6_k"]) if scheme == "q4_k" else scheme
    x = rng.choice(["f32", "bf16"])
    hidden = 256 * rng.randint(6, 18)
    inter = 256 * rng.randint(2 * hidden // 256, 3 * hidden // 256)
    # f32 prompts do three to four times the matrix work of bf16 ones
    m = _log_int(rng, 1, 900 if x == "f32" else 3000)
    y = "bf16" if x == "bf16" and m >= 64 else "f32"
    return _decoder(None, m, scheme, down, x, y, 2 if m < 64 else 1, hidden=hidden,
                    qkv=hidden + 256 * rng.randint(2, 8), inter=inter)


def _shapes(case):
    """(k, n, scheme) of the dense calls of one layer."""
    if case["kind"] == "linear":
        return [(case["k"], case["n"], case["scheme"])]
    h, i, s = case["hidden"], case["inter"], case["scheme"]
    return [(h, case["qkv"], s), (h, h, s), (h, 2 * i, s), (i, h, case["down"])]


# ---- inputs ----------------------------------------------------------------
def _f16_bytes(count, lo, hi, gen):
    v = torch.empty(count, device="cuda").uniform_(lo, hi, generator=gen).half()
    return v.view(torch.uint8).view(count, 2)


def _bytes(rows, count, gen):
    return torch.randint(0, 256, (rows, count), device="cuda", dtype=torch.uint8, generator=gen)


def _weights(scheme, n, k, gen):
    """Packed rows as a checkpoint holds them: uniform codes, scales of the
    sizes quantised layers have.  Returns (packed, scales, biases)."""
    if scheme == "q4_1":
        nb = n * (k // 32)
        return torch.cat([_f16_bytes(nb, 0.005, 0.05, gen), _f16_bytes(nb, -0.4, 0.0, gen), _bytes(nb, 16, gen)],
                         dim=1).view(-1), None, None
    if scheme == "q8_0":
        nb = n * (k // 32)
        q = torch.randint(-127, 128, (nb, 32), device="cuda", dtype=torch.int8, generator=gen).view(torch.uint8)
        return torch.cat([_f16_bytes(nb, 0.002, 0.02, gen), q], dim=1).view(-1), None, None
    if scheme == "q4_k":
        nb = n * (k // 256)
        return torch.cat([_f16_bytes(nb, 0.0005, 0.002, gen), _f16_bytes(nb, 0.0005, 0.005, gen),
                          _bytes(nb, 140, gen)], dim=1).view(-1), None, None
    if scheme == "q6_k":
        nb = n * (k // 256)
        sc = torch.randint(-64, 64, (nb, 16), device="cuda", dtype=torch.int8, generator=gen).view(torch.uint8)
        return torch.cat([_bytes(nb, 192, gen), sc, _f16_bytes(nb, 0.0002, 0.001, gen)], dim=1).view(-1), None, None
    g = k // _GROUP
    sc = torch.empty((n, g), device="cuda").uniform_(0.01, 0.1, generator=gen).to(torch.bfloat16)
    bi = torch.empty((n, g), device="cuda").uniform_(-0.5, 0.1, generator=gen).to(torch.bfloat16)
    return _bytes(n, k // 2, gen).view(-1), sc, bi


def _rows(m, k, dtype, gen):
    return torch.randn((m, k), device="cuda", generator=gen).to(dtype)


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "w8a8":
        m, k, n = case["m"], case["k"], case["n"]
        return {"x": _rows(m, k, torch.bfloat16, gen),
                "w": torch.randint(-127, 128, (k, n), device="cuda", dtype=torch.int8, generator=gen),
                "sw": torch.empty(n, device="cuda").uniform_(0.0005, 0.002, generator=gen)}
    if kind == "moe":
        e, h, i = case["experts"], case["hidden"], case["inter"]
        return {"gate_up": _weights(case["scheme"], e * 2 * i, h, gen)[0],
                "down": _weights(case["scheme"], e * h, i, gen)[0],
                "logits": torch.randn((case["m"], e), device="cuda", generator=gen),
                # (activations behind a norm, scaled so that the experts' outputs stay of order one)
                "x": (torch.randn((case["m"], h), device="cuda", generator=gen) * 0.1).to(_DT[case["x"]])}
    calls = []
    for _ in range(case.get("layers", 1)):
        for k, n, scheme in _shapes(case):
            w, sc, bi = _weights(scheme, n, k, gen)
            calls.append({"scheme": scheme, "k": k, "n": n, "w": w, "scales": sc, "biases": bi,
                          "x": _rows(case["m"], k, _DT[case["x"]], gen)})
    return {"calls": calls}


def prepare(case, seed):
    ctx = _context()
    s = {"case": case, "ctx": ctx, **_inputs(case, seed)}
    if case["kind"] == "w8a8":
        s["y"] = torch.empty((case["m"], case["n"]), device="cuda", dtype=torch.bfloat16)
    elif case["kind"] == "moe":
        s["act"] = torch.empty((case["m"] * case["top_k"], case["inter"]), device="cuda", dtype=_DT[case["x"]])
        s["y"] = torch.empty((case["m"], case["hidden"]), device="cuda")
    else:
        s["bound"] = []
        for c in s["calls"]:
            c["y"] = torch.empty((case["m"], c["n"]), device="cuda", dtype=_DT[case["y"]])
            s["bound"].append(ctx.bind_dequant_matmul(c["x"], c["w"], _SCHEME[c["scheme"]], c["n"], y=c["y"], stream=None,
                                                      group=_GROUP if c["scheme"] == "mlx4" else 32,
                                                      scales=c["scales"], biases=c["biases"]))
        s["y"] = [c["y"] for c in s["calls"]]
    return s


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "w8a8":
        return ctx.w8a8_gemm(state["x"], state["w"], state["sw"], case["n"], y=state["y"])
    if case["kind"] == "moe":
        scheme, e = _SCHEME[case["scheme"]], case["experts"]
        ids, probs = ctx.moe_route(state["logits"], case["top_k"], True)
        ctx.moe_grouped(state["x"], state["gate_up"], ids, probs, scheme, rlxq.MOE_EXPAND_SWIGLU, 2 * case["inter"], e,
                        y=state["act"])
        ctx.moe_grouped(state["act"], state["down"], ids, probs, scheme, rlxq.MOE_COMBINE, case["hidden"], e,
                        y=state["y"])
        return {"ids": ids, "probs": probs, "act": state["act"], "y": state["y"]}
    for call in state["bound"]:
        call()
    return state["y"]


# ---- what a pass cannot do without -----------------------------------------
def work(case):
    m = case["m"]
    if case["kind"] == "w8a8":
        k, n = case["k"], case["n"]
        return {"bytes": k * n + 4 * n + 2 * m * k + 2 * m * n, "flops": 2 * m * k * n}
    if case["kind"] == "moe":
        e, h, i, t, xs = case["experts"], case["hidden"], case["inter"], case["top_k"], _SIZE[case["x"]]
        fired = e * (1 - (1 - t / e) ** m)   # experts at least one token is routed to, expected
        return {"bytes": int(fired * 3 * h * i * _BPW[case["scheme"]] + m * (h * (xs + 4) + 2 * t * i * xs + 4 * e)),
                "flops": 6 * m * t * h * i}
    xs, ys = _SIZE[case["x"]], _SIZE[case["y"]]
    b = f = 0
    for k, n, scheme in _shapes(case):
        b += n * k * _BPW[scheme] + m * k * xs + m * n * ys
        f += 2 * m * n * k
    return {"bytes": int(b * case.get("layers", 1)), "flops": f * case.get("layers", 1)}


def tolerance(case):
    if case["kind"] == "w8a8":
        return {"rel": 8e-3}    # integer sums are exact; the output is rounded to bf16
    if case["kind"] == "moe":
        # bf16: the SwiGLU output is rounded to bf16 between the two grouped calls
        return {"rel": 3e-5 if case["x"] == "f32" else 8e-3, "max": 1e-3 if case["x"] == "f32" else 0.1, "differ": 1e-3}
    if case["y"] == "bf16":
        return {"rel": 1e-2, "max": 0.1}    # weights and output rounded to bf16
    # f32 sums; f32 rows of a few-row call are split into two bf16 halves (~2^-17 each)
    return {"rel": 2e-5, "max": 1e-3}


# ---- float64 ---------------------------------------------------------------
def _f16_at(blk, off):
    return blk[:, off:off + 2].contiguous().view(torch.float16).double()


def _six_bit_scales(q):
    """The 8 scales and 8 mins packed in the 12 bytes of a Q4_K super-block."""
    q = q.int()
    lo_s, lo_m = q[:, 0:4] & 63, q[:, 4:8] & 63
    hi_s = (q[:, 8:12] & 15) | ((q[:, 0:4] >> 6) << 4)
    hi_m = (q[:, 8:12] >> 4) | ((q[:, 4:8] >> 6) << 4)
    return torch.cat([lo_s, hi_s], 1).double(), torch.cat([lo_m, hi_m], 1).double()


def _dequant(scheme, w, n, k, scales=None, biases=None):
    if scheme == "q4_1":
        b = w.view(n * (k // 32), 20)
        q = torch.cat([b[:, 4:] & 15, b[:, 4:] >> 4], 1).double()
        return (q.mul_(_f16_at(b, 0)).add_(_f16_at(b, 2))).view(n, k)
    if scheme == "q8_0":
        b = w.view(n * (k // 32), 34)
        return b[:, 2:].contiguous().view(torch.int8).double().mul_(_f16_at(b, 0)).view(n, k)
    if scheme == "q4_k":
        b = w.view(n * (k // 256), 144)
        sc, mn = _six_bit_scales(b[:, 4:16])
        q = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()   # 64-weight groups: low, then high nibbles
        return (q.mul_((_f16_at(b, 0) * sc)[:, :, None]).sub_((_f16_at(b, 2) * mn)[:, :, None])).view(n, k)
    if scheme == "q6_k":
        b = w.view(n * (k // 256), 210)
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(-1, 2, 4, 2, 1)
        low = torch.cat([ql & 15, ql >> 4], 2)                            # quarter j: ql half j & 1, nibble j >> 1
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (high << 4)).double().sub_(32).view(-1, 2, 4, 2, 16)
        return q.mul_(sc).view(-1, 256).mul_(_f16_at(b, 208)).view(n, k)
    b = w.view(n, k // 2)
    q = torch.stack([b & 15, b >> 4], 2).view(n, k // _GROUP, _GROUP).double()   # eight codes a word, low nibble first
    return q.mul_(scales.double()[:, :, None]).add_(biases.double()[:, :, None]).view(n, k)


def exact(case, seed):
    d = _inputs(case, seed)
    if case["kind"] == "w8a8":
        x = d["x"].float()
        s = x.abs().amax(dim=1, keepdim=True) / 127.0     # the quantiser's own rounding, in f32
        s = torch.where(s > 0, s, torch.ones_like(s))
        v = x * (1.0 / s)
        q = torch.clamp(torch.sign(v) * torch.floor(v.abs() + 0.5), -127, 127).double()
        return (q @ d["w"].double()) * s.double() * d["sw"].double()
    if case["kind"] == "moe":
        e, h, i, t = case["experts"], case["hidden"], case["inter"], case["top_k"]
        p, ids = torch.topk(torch.softmax(d["logits"].double(), 1), t, dim=1)
        p = p / p.sum(1, keepdim=True)
        x = d["x"].double()
        act = torch.zeros((case["m"], t, i), device="cuda", dtype=torch.float64)
        y = torch.zeros((case["m"], h), device="cuda", dtype=torch.float64)
        rb_g, rb_d = d["gate_up"].numel() // e, d["down"].numel() // e
        for ex in range(e):
            r, j = (ids == ex).nonzero(as_tuple=True)
            if not r.numel():
                continue
            gu = x[r] @ _dequant(case["scheme"], d["gate_up"][ex * rb_g:(ex + 1) * rb_g], 2 * i, h).T
            a = gu[:, :i] * torch.sigmoid(gu[:, :i]) * gu[:, i:]
            act[r, j] = a
            y.index_add_(0, r, p[r, j][:, None] * (a @ _dequant(case["scheme"], d["down"][ex * rb_d:(ex + 1) * rb_d], h, i).T))
        return {"ids": None, "probs": p, "act": act.view(-1, i), "y": y}
    out = []
    for c in d["calls"]:
        w = _dequant(c["scheme"], c["w"], c["n"], c["k"], c["scales"], c["biases"])
        out.append(c["x"].double() @ w.T)
    return out
