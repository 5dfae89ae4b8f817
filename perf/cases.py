"""The calls a DiT forward makes of this package, as timed cases.

A denoising step of the model runs, per block and per stream (image tokens, text tokens),
LayerNorm + AdaLN, FP8 Linears (per-token quantization and the row-wise scaled GEMM), the
QK norm with 3D rotary embedding, the gated residual with the next norm, and the MLP; the
streaming runtime adds the pre-RoPE K stage, the K ring cache and the KV-pool commit. Each
listed case is one such call (the MLP: the chain a block makes of them) through
joyomni_ops / joyomni_ops.dit_ops at the shapes of the package's workloads: hidden 4096
with 32 heads and 1560 tokens a latent frame, hidden 3072 with 24 heads and 3510 tokens a
frame, and a text prompt of tens to hundreds of tokens. draw() spreads the same calls over
their ranges of tokens, widths, heads, batches, data types and options.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_root, "joyai-video-edit_amd"))

import joyomni_ops as jo  # noqa: E402
from joyomni_ops import dit_ops  # noqa: E402

FP8 = torch.float8_e4m3fn
FP8_MAX = 448.0
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed() -> list:
    return [
        # The text stream's q and k norm (a torch RMSNorm module in the model) on a short
        # prompt's packed qkv: the smallest call of a block.
        dict(name="text_qk_norm", kind="qk_norm", B=1, L=77, H=32, D=128, dtype="bf16"),
        # LayerNorm + AdaLN of the image stream, per-sample modulation.
        dict(name="image_ln_modulate", kind="ln_modulate", B=1, L=3120, N=4096, dtype="bf16",
             per_token=False, affine=False),
        # The image stream's QK norm + RoPE: slices of the packed qkv in, contiguous q and k
        # out, the model's fp32 tables.
        dict(name="image_qk_rope", kind="qk_rope", B=1, L=3120, H=32, D=128, gh=30, gw=52),
        # The KV store forward of one frame: q and k rotated in place, K before RoPE staged.
        dict(name="store_qk_stage", kind="qk_stage", B=1, L=1560, H=32, D=128, gh=30, gw=52),
        # QK norm + RoPE of a three-frame chunk with K written to the ring cache.
        dict(name="ring_qk_chunk", kind="qk_ring", B=1, frames=3, H=24, D=128, gh=45, gw=78,
             slots=7, t0=21),
        # Per-block RMSNorm -> FP8 of a ragged token count.
        dict(name="rmsnorm_fp8_block", kind="rms_quant", M=4725, N=3072, group=128,
             dtype="bf16"),
        # Gated residual + LayerNorm + AdaLN -> FP8 of a three-frame chunk.
        dict(name="chunk_add_norm_fp8", kind="add_norm_fp8", B=1, L=10530, N=3072,
             dtype="bf16"),
        # The text stream's qkv projection on a short prompt (quantization + GEMM).
        dict(name="text_linear_qkv", kind="linear", B=1, L=77, K=4096, N=12288, bias=True,
             dtype="bf16"),
        # The image stream's attention output projection (quantization + GEMM).
        dict(name="image_linear_out", kind="linear", B=1, L=3120, K=4096, N=4096, bias=True,
             dtype="bf16"),
        # The text stream's MLP, a prompt of 256 tokens.
        dict(name="text_mlp", kind="mlp", B=1, L=256, K=4096, F=16384),
        # The image stream's MLP: the largest part of a block.
        dict(name="image_mlp", kind="mlp", B=1, L=3120, K=4096, F=16384),
        # The KV-pool commit of one frame for all 40 layers.
        dict(name="kv_commit", kind="kv_commit", layers=40, B=1, T=1560, P=3120, off=1560, H=32,
             D=128),
    ]


# ---------------------------------------------------------------------------
# Drawn cases.
# ---------------------------------------------------------------------------
def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo: int, hi: int, unit: int = 16) -> int:
    """A hidden width: mostly a multiple of 128, some of 64, some ragged (multiples of unit)."""
    u = rng.choice((128, 128, 128, 128, 128, 64, 64, unit))
    return max(lo, _log(rng, lo, hi) // u * u)


def draw(rng) -> dict:
    kind = rng.choice(("qk_norm", "ln_modulate", "qk_rope", "qk_stage", "qk_ring", "rms_quant",
                       "add_norm_fp8", "linear", "linear", "mlp", "kv_commit"))
    half = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    B = rng.choice((1, 1, 1, 2))
    H = rng.choice((8, 12, 16, 24, 24, 32, 32, rng.randint(5, 40)))
    D = rng.choice((64, 128, 128, 128, 256))
    H = max(1, min(H, 5120 // D))
    gh, gw = rng.randint(11, 45), rng.randint(20, 78)
    frames = rng.randint(1, 3)
    if kind == "qk_norm":
        return dict(kind=kind, B=B, L=_log(rng, 1, 4096), H=H, D=D, dtype=half)
    if kind == "ln_modulate":
        return dict(kind=kind, B=B, L=_log(rng, 1, 10530) // B + 1, N=_width(rng, 768, 8192, 4),
                    dtype=rng.choice((half, half, "fp32")), per_token=rng.random() < 0.25,
                    affine=rng.random() < 0.25)
    if kind in ("qk_rope", "qk_stage"):
        return dict(kind=kind, B=B, L=frames * gh * gw, H=H, D=D, gh=gh, gw=gw)
    if kind == "qk_ring":
        return dict(kind=kind, B=B, frames=frames, H=H, D=D, gh=gh, gw=gw,
                    slots=frames + rng.randint(0, 5), t0=rng.randint(0, 200))
    if kind == "rms_quant":
        group = rng.choice((0, 128))
        return dict(kind=kind, M=_log(rng, 1, 10530), N=_width(rng, 768, 8192, 128 if group else 8),
                    group=group, dtype=half)
    if kind == "add_norm_fp8":
        return dict(kind=kind, B=B, L=_log(rng, 1, 10530) // B + 1, N=_width(rng, 768, 8192, 8),
                    dtype=half)
    if kind == "linear":
        return dict(kind=kind, B=B, L=_log(rng, 1, 4096) // B + 1, K=_width(rng, 1024, 8192),
                    N=_width(rng, 1024, 12288), bias=rng.random() < 0.75, dtype=half)
    if kind == "mlp":
        K = _width(rng, 1024, 4096)
        return dict(kind=kind, B=B, L=_log(rng, 16, 3000) // B + 1, K=K,
                    F=_width(rng, 2 * K, 4 * K))
    T = _log(rng, 64, 1560)
    off = rng.randint(0, 2) * T
    return dict(kind=kind, layers=_log(rng, 1, 40), B=1, T=T, P=off + T + rng.randint(0, T),
                off=off, H=H, D=D)


# ---------------------------------------------------------------------------
# Inputs (from the seed alone, plain torch).
# ---------------------------------------------------------------------------
def _rope_dims(D: int) -> tuple:
    """t / h / w rotary sizes, in the ratio of the model's (44, 42, 42) at head_dim 128."""
    hw = D * 42 // 128 // 2 * 2
    return (D - 2 * hw, hw, hw)


def _grid_angles(tokens: int, D: int, gh: int, gw: int, t0: int, device) -> torch.Tensor:
    """fp32 [tokens, D/2] rotation angles pos * 1/10000^(2j/dim) of the t, h, w axes."""
    n = torch.arange(tokens, device=device)
    pos = (t0 + n // (gh * gw), n % (gh * gw) // gw, n % gw)
    cols = []
    for p, d in zip(pos, _rope_dims(D)):
        f = 1.0 / (10000.0 ** (torch.arange(0, d, 2)[: d // 2].float() / d))
        cols.append(p.float()[:, None] * f.to(device)[None, :])
    return torch.cat(cols, 1)


def _tables(ang: torch.Tensor) -> tuple:
    """(cos, sin) fp32 [1, tokens, D], each value repeated for the two elements of its pair."""
    return tuple(t.repeat_interleave(2, 1).unsqueeze(0).contiguous()
                 for t in (ang.cos(), ang.sin()))


def _weight(n: int, k: int, g, dev) -> torch.Tensor:
    return (torch.randn(n, k, generator=g, device=dev) * k ** -0.5).to(torch.bfloat16)


def _inputs(c: dict, seed: int) -> dict:
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(seed)

    def rand(*shape, mul=1.0, add=0.0, dtype=torch.bfloat16):
        x = torch.randn(*shape, generator=g, device=dev)
        return (x.mul_(mul).add_(add) if (mul, add) != (1.0, 0.0) else x).to(dtype)

    def hidden(*shape, dtype):
        """Activations with the outliers a transformer's hidden states show."""
        x = torch.randn(*shape, generator=g, device=dev)
        big = torch.rand(*shape, generator=g, device=dev) < 0.005
        return torch.where(big, 40 * x, x).to(dtype)

    kind, dt = c["kind"], DTYPES[c.get("dtype", "bf16")]
    if kind in ("qk_norm", "qk_rope", "qk_stage", "qk_ring"):
        L = c["frames"] * c["gh"] * c["gw"] if kind == "qk_ring" else c["L"]
        D = c["D"]
        t = {"qkv": rand(c["B"], L, 3, c["H"], D, dtype=dt),
             "qw": rand(D, mul=0.1, add=1.0, dtype=dt), "kw": rand(D, mul=0.1, add=1.0, dtype=dt)}
        if kind in ("qk_rope", "qk_stage"):
            t["cos"], t["sin"] = _tables(_grid_angles(L, D, c["gh"], c["gw"], 0, dev))
        if kind == "qk_stage":
            t["stage"] = torch.zeros(c["B"], L, c["H"], D, dtype=dt, device=dev)
        if kind == "qk_ring":
            t["cache"] = torch.zeros(c["B"], c["slots"] * c["gh"] * c["gw"] * c["H"], D, dtype=dt,
                                     device=dev)
        return t
    if kind in ("ln_modulate", "add_norm_fp8"):
        B, L, N = c["B"], c["L"], c["N"]
        mod = (B, L, N) if c.get("per_token") else (B, N)
        t = {"x": rand(B, L, N, dtype=dt), "shift": rand(*mod, mul=0.2, dtype=dt),
             "scale": rand(*mod, mul=0.2, dtype=dt)}
        if kind == "add_norm_fp8":
            t["residual"] = rand(B, L, N, dtype=dt)
            t["gate"] = rand(*mod, mul=0.2, dtype=dt)
        if c.get("affine"):
            t["weight"] = rand(N, mul=0.1, add=1.0, dtype=dt)
            t["bias"] = rand(N, mul=0.1, dtype=dt)
        return t
    if kind == "rms_quant":
        return {"x": hidden(c["M"], c["N"], dtype=dt),
                "weight": rand(c["N"], mul=0.1, add=1.0, dtype=dt)}
    if kind == "linear":
        return {"x": hidden(c["B"], c["L"], c["K"], dtype=dt), "w": _weight(c["N"], c["K"], g, dev),
                "bias": rand(c["N"], mul=0.02, dtype=dt) if c["bias"] else None}
    if kind == "mlp":
        B, L, K, F = c["B"], c["L"], c["K"], c["F"]
        t = {"x": rand(B, L, K)}
        for name in ("shift", "scale", "gate"):
            t[name] = rand(B, K, mul=0.2)
        t["up"], t["up_bias"] = _weight(F, K, g, dev), rand(F, mul=0.02)
        t["down"], t["down_bias"] = _weight(K, F, g, dev), rand(K, mul=0.02)
        return t
    shape = (c["layers"], c["B"], c["T"], c["H"], c["D"])
    pool = (c["layers"], c["B"], c["P"], c["H"], c["D"])
    t = {"stage_k": rand(*shape), "stage_v": rand(*shape),
         "pool_k": torch.zeros(pool, dtype=dt, device=dev),
         "pool_v": torch.zeros(pool, dtype=dt, device=dev)}
    t["cos"], t["sin"] = _tables(_grid_angles(c["T"], c["D"], 30, 52, 0, dev))
    return t


def prepare(case: dict, seed: int) -> dict:
    t = _inputs(case, seed)
    t["case"] = case
    kind = case["kind"]
    if kind == "linear":
        t["w"] = dit_ops.quantize_weight_per_channel(t["w"])
    elif kind == "mlp":
        t["up"] = dit_ops.quantize_weight_per_channel(t["up"])
        t["down"] = dit_ops.quantize_weight_per_channel(t["down"])
    elif kind == "qk_ring":
        t["freqs"] = jo.rope_freqs(case["D"], _rope_dims(case["D"]), 10000.0)
    elif kind == "rms_quant":
        # The FP8 operand buffers that the next GEMM reads, kept by the caller.
        M, N, group = case["M"], case["N"], case["group"]
        t["q"] = torch.empty(M, N, dtype=FP8, device="cuda")
        t["s"] = torch.empty((M, N // group) if group else (M, 1), device="cuda")
    return t


def run(t: dict):
    c = t["case"]
    kind = c["kind"]
    if kind == "qk_norm":
        qkv = t["qkv"]
        return (dit_ops.rms_norm_module(qkv[:, :, 0], t["qw"], EPS),
                dit_ops.rms_norm_module(qkv[:, :, 1], t["kw"], EPS))
    if kind == "ln_modulate":
        return dit_ops.fused_layernorm_modulate(t["x"], t["shift"], t["scale"],
                                                weight=t.get("weight"), bias=t.get("bias"), eps=EPS)
    if kind == "qk_rope":
        qkv = t["qkv"]
        return dit_ops.fused_qk_norm_rope_3d(qkv[:, :, 0], qkv[:, :, 1], t["qw"], t["kw"],
                                             (t["cos"], t["sin"]), eps=EPS)
    if kind == "qk_stage":
        qkv = t["qkv"]
        return dit_ops.fused_qk_norm_rope_3d_kstage(qkv[:, :, 0], qkv[:, :, 1], t["qw"], t["kw"],
                                                    (t["cos"], t["sin"]), eps=EPS,
                                                    k_stage=t["stage"])
    if kind == "qk_ring":
        qkv, D, gh, gw = t["qkv"], c["D"], c["gh"], c["gw"]
        q = qkv[:, :, 0]
        jo.fused_qk_norm_rope_3d_kvcache(q, qkv[:, :, 1], t["cache"], c["frames"] * gh * gw, c["H"],
                                         EPS, t["qw"], t["kw"], t["freqs"], _rope_dims(D), (gh, gw),
                                         c["t0"], jo.kv_ring_slot(c["t0"], c["frames"], c["slots"]))
        return q, t["cache"]
    if kind == "rms_quant":
        jo.rmsnorm_quant_fp8(t["x"], t["weight"], EPS, t["q"], t["s"], c["group"])
        return t["q"], t["s"]
    if kind == "add_norm_fp8":
        return dit_ops.fused_add_gate_layernorm_modulate_fp8(t["residual"], t["x"], t["gate"],
                                                             t["shift"], t["scale"], eps=EPS)
    if kind == "linear":
        return dit_ops.fp8_linear(t["x"], *t["w"], t["bias"], t["x"].dtype)
    if kind == "mlp":
        x = t["x"]
        x_q, x_s = dit_ops.layernorm_modulate_fp8(x, t["shift"], t["scale"], eps=EPS)
        h = dit_ops.fp8_linear_quantized(x_q, x_s, *t["up"], t["up_bias"])
        h_q, h_s = dit_ops.gelu_quantize_activation_fp8(h)
        y = dit_ops.fp8_linear_quantized(h_q, h_s, *t["down"], t["down_bias"])
        return dit_ops.fused_add_gate(x, y.view_as(x), t["gate"])
    dit_ops.commit_kv_pool(t["pool_k"], t["pool_v"], t["stage_k"], t["stage_v"], c["off"], t["cos"],
                           t["sin"])
    return t["pool_k"], t["pool_v"]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is.
# ---------------------------------------------------------------------------
def work(c: dict) -> dict:
    kind = c["kind"]
    e = {"fp32": 4}.get(c.get("dtype"), 2)  # bytes of an activation element
    if kind in ("qk_norm", "qk_rope", "qk_stage", "qk_ring"):
        tokens = c["B"] * (c["frames"] * c["gh"] * c["gw"] if kind == "qk_ring" else c["L"])
        rows = tokens * c["H"] * c["D"] * 2
        n = {"qk_norm": 4, "qk_rope": 4, "qk_stage": 5, "qk_ring": 4}[kind] * rows
        if kind in ("qk_rope", "qk_stage"):
            n += 2 * c["L"] * c["D"] // 2 * 4  # one cos and one sin a pair
        return {"bytes": n + 4 * c["D"], "flops": 10.0 * tokens * c["H"] * c["D"] * 2}
    if kind == "ln_modulate":
        rows = c["B"] * c["L"] * c["N"] * e
        mod = rows if c["per_token"] else c["B"] * c["N"] * e
        return {"bytes": 2 * rows + 2 * mod, "flops": 8.0 * rows / e}
    if kind == "add_norm_fp8":
        n = c["B"] * c["L"] * c["N"]
        return {"bytes": n * (3 * e + 1) + 4 * c["B"] * c["L"] + 3 * c["B"] * c["N"] * e,
                "flops": 12.0 * n}
    if kind == "rms_quant":
        n = c["M"] * c["N"]
        return {"bytes": 3 * n + 4 * (n // c["group"] if c["group"] else c["M"]) + 2 * c["N"],
                "flops": 6.0 * n}
    if kind == "linear":
        M, K, N = c["B"] * c["L"], c["K"], c["N"]
        return {"bytes": M * K * 2 + N * K + N * 4 + M * N * 2 + (N * 2 if c["bias"] else 0),
                "flops": 2.0 * M * N * K}
    if kind == "mlp":
        M, K, F = c["B"] * c["L"], c["K"], c["F"]
        return {"bytes": 2 * M * K * 2 + 2 * K * F + 6 * (K + F) + 6 * c["B"] * K,
                "flops": 4.0 * M * K * F}
    n = c["layers"] * c["B"] * c["T"] * c["H"] * c["D"]
    return {"bytes": 8 * n + 2 * c["T"] * c["D"] // 2 * 4, "flops": 3.0 * n}


def tolerance(c: dict) -> dict:
    """About four times the distance measured between the path and exact() below."""
    kind = c["kind"]
    if kind in ("rms_quant", "add_norm_fp8"):
        # FP8 codes: the few that fall on the other side of a rounding boundary are one
        # code (an eighth of the value) apart; the bf16 residual beside them.
        return {"rel": 8e-3, "max": 0.15}
    if kind == "mlp":
        # A value of the hidden layer that rounds to the other FP8 code moves a whole row.
        return {"rel": 8e-3, "max": 0.1}
    if c.get("dtype") == "fp16":
        return {"rel": 1e-3, "max": 4e-3}
    if c.get("dtype") == "fp32":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 8e-3, "max": 0.04}  # one rounding to bf16


# ---------------------------------------------------------------------------
# The same in 64 bits (values that a call stores in 16 or 8 bits on its way, and
# normalizes or multiplies after that, are rounded there).
# ---------------------------------------------------------------------------
def _quant(x: torch.Tensor, dim: int = -1) -> tuple:
    """(codes, scale) of rows: scale = max / 448 in fp32, codes = e4m3(x / scale)."""
    s = (x.abs().amax(dim, keepdim=True).float() / FP8_MAX).double()
    inv = torch.where(s == 0, torch.zeros_like(s), 1.0 / s)
    q = (x * inv).clamp(-FP8_MAX, FP8_MAX).float().to(FP8)
    return q.double(), s


def _weight_codes(w: torch.Tensor) -> tuple:
    """Per-channel codes [N, K] and fp32 scales [N] of a bf16 weight."""
    s = w.float().abs().amax(1).clamp_min(1e-8) / FP8_MAX
    return (w.float() / s[:, None]).clamp(-FP8_MAX, FP8_MAX).to(FP8).double(), s.double()


def _linear(x: torch.Tensor, w: torch.Tensor, bias) -> torch.Tensor:
    """An FP8 Linear of x [M, K] (16-bit values held in 64)."""
    q, s = _quant(x)
    wq, ws = _weight_codes(w)
    y = (q @ wq.t()) * ws * s
    return y if bias is None else y + bias.double()


def _ln_mod(x, shift, scale, weight=None, bias=None):
    mu = x.mean(-1, keepdim=True)
    y = (x - mu) / ((x - mu).square().mean(-1, keepdim=True) + EPS).sqrt()
    if weight is not None:
        y = y * weight.double() + bias.double()
    wide = (lambda m: m.double() if m.dim() == 3 else m.double().unsqueeze(1))  # noqa: E731
    return y * (1 + wide(scale)) + wide(shift)


def _rms(x, weight):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * weight.double()


def _rotate(x, cos, sin):
    """Interleaved pairs of x [B, L, H, D] by cos, sin [L, D/2]."""
    a, b = x[..., 0::2], x[..., 1::2]
    c, s = cos[None, :, None, :], sin[None, :, None, :]
    return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)


def exact(case: dict, seed: int):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "qk_norm":
        # The module rounds the normalized row to its type before the weight.
        def module(x, w):
            x = x.double()
            n = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()
            return n.to(w.dtype).double() * w.double()
        return module(t["qkv"][:, :, 0], t["qw"]), module(t["qkv"][:, :, 1], t["kw"])
    if kind == "ln_modulate":
        return _ln_mod(t["x"].double(), t["shift"], t["scale"], t.get("weight"), t.get("bias"))
    if kind in ("qk_rope", "qk_stage"):
        # The tables are read as bf16.
        cos, sin = (x[0, :, ::2].to(torch.bfloat16).double() for x in (t["cos"], t["sin"]))
        q, k = _rms(t["qkv"][:, :, 0].double(), t["qw"]), _rms(t["qkv"][:, :, 1].double(), t["kw"])
        out = _rotate(q, cos, sin), _rotate(k, cos, sin)
        return out + (k,) if kind == "qk_stage" else out
    if kind == "qk_ring":
        gh, gw, frames, slots = case["gh"], case["gw"], case["frames"], case["slots"]
        ang = _grid_angles(frames * gh * gw, case["D"], gh, gw, case["t0"], "cuda").double()
        q, k = (_rotate(_rms(t["qkv"][:, :, i].double(), t[w]), ang.cos(), ang.sin())
                for i, w in ((0, "qw"), (1, "kw")))
        cache = t["cache"].double().view(case["B"], slots, gh * gw, case["H"], case["D"])
        first = case["t0"] // frames % slots
        for f in range(frames):
            cache[:, (first + f) % slots] = k[:, f * gh * gw:(f + 1) * gh * gw]
        return q, cache.view(t["cache"].shape)
    if kind == "rms_quant":
        y = _rms(t["x"].double(), t["weight"])
        if case["group"]:
            q, s = _quant(y.view(case["M"], -1, case["group"]))
            return q.view(y.shape), s.squeeze(-1)
        return _quant(y)
    if kind == "add_norm_fp8":
        # The residual is rounded once, and what is stored is what is normalized.
        r = t["residual"].double() + t["x"].double() * t["gate"].double().unsqueeze(1)
        dt = t["x"].dtype
        y = _ln_mod(r.to(dt).double(), t["shift"], t["scale"]).to(dt).double()
        q, s = _quant(y.view(-1, case["N"]))
        return r, q, s
    if kind == "linear":
        return _linear(t["x"].view(-1, case["K"]).double(), t["w"], t["bias"]).view(
            case["B"], case["L"], -1)
    if kind == "mlp":
        x, bf = t["x"].double(), torch.bfloat16
        y = _ln_mod(x, t["shift"], t["scale"]).to(bf).double().view(-1, case["K"])
        h = _linear(y, t["up"], t["up_bias"]).to(bf).double()
        h = (0.5 * h * (1 + torch.tanh(math.sqrt(2 / math.pi) * (h + 0.044715 * h ** 3))))
        y = _linear(h.to(bf).double(), t["down"], t["down_bias"]).to(bf).double()
        return x + y.view(x.shape) * t["gate"].double().unsqueeze(1)
    off, T = case["off"], case["T"]
    pk, pv = t["pool_k"].double(), t["pool_v"].double()
    cos, sin = t["cos"][0, :, ::2].double(), t["sin"][0, :, ::2].double()
    for i in range(case["layers"]):
        pk[i, :, off:off + T] = _rotate(t["stage_k"][i].double(), cos, sin)
        pv[i, :, off:off + T] = t["stage_v"][i].double()
    return pk, pv
