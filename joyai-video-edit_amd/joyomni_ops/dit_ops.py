"""DiT-side call shims over joyomni_ops, with the reference's names and signatures.

Counterpart of deploy/xvideo/models/dit/sgl_fused_ops.py:1-117 (the functions
MMDoubleStreamBlock.forward calls, dit.py:351-476) and of the activation
quantization step of Fp8Linear.forward (deploy/xvideo/models/dit/fp8_linear.py:138-169).
Same arguments, same results; the differences are in the HBM traffic:

  fused_layernorm_modulate  reads per-sample shift/scale [B, D] in place, one
                            row per sample, instead of materialising [B*L, D]
                            copies (sgl_fused_ops.py:44-51 expands and copies them).
  fused_qk_norm_rope_3d     identical contract; strided q/k slices and fp32 tables are
                            read as they are and the rotated rows written once
                            (sgl_fused_ops.py:73-94 copies q/k and halves, copies and
                            casts the tables first).
  rmsnorm_qk_bf16           normalizes the K slice of the packed qkv in place of
                            its .contiguous() copy (sgl_fused_ops.py:108).

Additional entry points for callers that can use the new fused ops:

  fused_qk_norm_rope_3d_grid_views  RMSNorm + RoPE in place on q/k views of the
                            packed qkv [B, L, 3, H, D] with angles computed from
                            grid positions (no tables, no .contiguous() copies).
  fused_qk_norm_rope_3d_kstage  the pre-RoPE K-cache path of dit.py:360-370
                            (rmsnorm_qk_bf16 of K, then fused_qk_norm_rope_3d) in one
                            pass that reads K once; q / k rotated in place on their
                            packed-qkv views (no .contiguous() copies).
  fused_add_gate_layernorm_modulate residual + x * gate and the following
                            fused_layernorm_modulate in one pass (dit.py:447-457).
  quantize_activation_fp8   x_q, x_scale of Fp8Linear.forward (fp8_linear.py:140-166).
  layernorm_modulate_fp8    fused_layernorm_modulate followed by that quantization,
                            in one pass (the bf16 output is never written).
  fused_add_gate_layernorm_modulate_fp8  the same after residual + x * gate.
  commit_kv_pool            StreamingGraphRunner.run_commit (graph_runner.py:137-142)
                            for all layers in one launch.
  rms_norm_module           the torch RMSNorm module's forward (dit.py:244-249) that
                            the text stream applies to q and k (dit.py:384-385),
                            read from the packed qkv view.
  gelu_quantize_activation_fp8  the MLP activation gelu(h, approximate="tanh")
                            (dit.py:91-92, 433) and the quantization of the
                            following Fp8Linear.forward in one pass (the bf16
                            activation is never written).
  fp8_linear                Fp8Linear.forward (fp8_linear.py:155-169): per-token
                            quantization + fp8_scaled_mm; quantize_weight_per_channel
                            is its weight preparation (fp8_linear.py:100-110).
"""
from __future__ import annotations

from typing import Optional, Sequence, Tuple

import torch

from . import (fp8_scaled_mm, fused_add_layernorm_scale_shift, fused_qk_norm_rope_3d_grid,
               kv_commit_rope, rope_freqs)

# One dispatch per call: the reshapes, output allocations and launches of these
# calls are made inside the op (at a few rows they are what a call costs: an
# Fp8Linear of 12 rows 16 us from Python, its two kernels 6).
_ops = torch.ops.joyomni_ops
_quantize_activation = _ops.quantize_activation.default
_gelu_quantize_activation = _ops.gelu_quantize_activation.default
_fp8_linear = _ops.fp8_linear.default
_layernorm_modulate = _ops.layernorm_modulate.default
_add_gate_layernorm_modulate_fp8 = _ops.add_gate_layernorm_modulate_fp8.default
_rmsnorm_last = _ops.rmsnorm_last.default
_qk_norm_rope_inplace = _ops.qk_norm_rope_inplace.default
_qk_norm_rope_copies = _ops.qk_norm_rope_copies.default
_qk_norm_rope_kstage = _ops.qk_norm_rope_kstage.default


# Shapes of the results, for tracing (torch.compile and fake tensors), of the ops
# that allocate outputs whose calls traced when the Python shims allocated them;
# the ops that only write into their arguments need none.
@torch.library.register_fake("joyomni_ops::quantize_activation")
@torch.library.register_fake("joyomni_ops::gelu_quantize_activation")
def _(x):
    K = x.shape[-1]
    M = x.numel() // K
    return x.new_empty((M, K), dtype=torch.float8_e4m3fn), x.new_empty((M, 1), dtype=torch.float32)


@torch.library.register_fake("joyomni_ops::add_gate_layernorm_modulate_fp8")
def _(x, residual, gate, gamma, beta, scale, shift, eps):
    B, L, D = x.shape
    return (x.new_empty((B * L, D), dtype=torch.float8_e4m3fn),
            x.new_empty((B * L, 1), dtype=torch.float32))


@torch.library.register_fake("joyomni_ops::qk_norm_rope_copies")
def _(q, k, eps, q_weight, k_weight, cos, sin):
    return q.new_empty(q.shape), k.new_empty(k.shape)


def available() -> bool:
    """The reference's availability probe (sgl_fused_ops.py:14-27): the ops load at import."""
    return True


def fused_layernorm_modulate(
    x: torch.Tensor,
    shift: torch.Tensor,
    scale: torch.Tensor,
    *,
    weight: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
) -> torch.Tensor:
    """LayerNorm(x; weight, bias) * (1 + scale) + shift for x [B, L, D]
    (sgl_fused_ops.py:30-54). shift/scale: [B, D], [B, 1, D] or [B, L, D].

    Per-sample vectors are read in place, one row per sample of L tokens
    (fused_norm_scale_shift_per_sample), for any B: no [B*L, D] expanded
    copies; per-token modulation is read a row each."""
    return _layernorm_modulate(x, weight, bias, scale, shift, eps)


def fused_qk_norm_rope_3d(
    q: torch.Tensor,
    k: torch.Tensor,
    q_norm_weight: torch.Tensor,
    k_norm_weight: torch.Tensor,
    freqs_cis: Tuple[torch.Tensor, torch.Tensor],
    *,
    eps: float = 1e-6,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per-head RMSNorm + interleaved RoPE of q, k [B, L, H, D] from
    (cos, sin) tables [1, L, D] or [L, D/2] (sgl_fused_ops.py:57-99). Returns
    contiguous (q, k): copies when q / k are strided views (such as the slices
    of a packed qkv), which leaves the inputs untouched; q / k themselves,
    rotated in place, when they are already contiguous (.contiguous() is then
    a no-op), as in the reference."""
    if q.dtype != torch.bfloat16:
        raise RuntimeError(f"fused_qk_norm_rope_3d requires bf16 q/k, got {q.dtype}")
    B, L, H, D = q.shape
    cos, sin = freqs_cis
    qw, kw = _bf16(q_norm_weight), _bf16(k_norm_weight)
    if (q.is_contiguous() or k.is_contiguous()
            or (torch.is_grad_enabled() and (q.requires_grad or k.requires_grad))):
        q = q.contiguous()  # outside the op: autograd records the copies
        k = k.contiguous()
        _qk_norm_rope_inplace(q, k, eps, qw, kw, cos, sin)
        return q, k
    # Strided slices and fp32 tables: one pass from where they are
    # ([1, 3120, 32, 128] of a packed qkv: 50.4 -> 19.3 us on MI355X against
    # the copies of q and k, the four table kernels and the paired op).
    return _qk_norm_rope_copies(q, k, eps, qw, kw, cos, sin)


def _bf16(w: torch.Tensor) -> torch.Tensor:
    return w if w.dtype is torch.bfloat16 else w.to(torch.bfloat16)


def fused_qk_norm_rope_3d_kstage(
    q: torch.Tensor,
    k: torch.Tensor,
    q_norm_weight: torch.Tensor,
    k_norm_weight: torch.Tensor,
    freqs_cis: Tuple[torch.Tensor, torch.Tensor],
    *,
    eps: float = 1e-6,
    k_stage: Optional[torch.Tensor] = None,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """The K-cache-before-RoPE branch of MMDoubleStreamBlock.forward
    (dit.py:360-370): k_for_cache = rmsnorm_qk_bf16(k, k_norm_weight) and
    q, k = fused_qk_norm_rope_3d(q, k, ...), in one pass that reads K once.

    q, k: bf16 [B, L, H, D], typically the q / k slices of the packed qkv
    [B, L, 3, H, D] (heads contiguous per token); they are normalized and
    rotated IN PLACE and returned (the reference returns rotated contiguous
    copies and leaves the qkv slices as they were; the DiT forward reads only
    the returned q, k and the v slice afterwards). freqs_cis: (cos, sin) of
    [1, L, D] or [L, D/2]. k_stage: bf16 [B, L, H, D] destination of the
    pre-RoPE normalized K (e.g. a layer's slice of the graph runner's stage
    buffer), allocated when None. Returns (q, k, k_stage); k_stage equals
    rmsnorm_qk_bf16(k) of the input k bit for bit."""
    if q.dtype != torch.bfloat16 or k.dtype != torch.bfloat16:
        raise RuntimeError(f"fused_qk_norm_rope_3d_kstage requires bf16 q/k, got {q.dtype}")
    B, L, H, D = q.shape
    if k_stage is None:
        k_stage = torch.empty((B, L, H, D), dtype=torch.bfloat16, device=q.device)
    cos, sin = freqs_cis
    _qk_norm_rope_kstage(q, k, k_stage, eps, _bf16(q_norm_weight).contiguous(),
                         _bf16(k_norm_weight).contiguous(), cos, sin)
    return q, k, k_stage


def rmsnorm_qk_bf16(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    """RMSNorm over the last dim of a bf16 tensor (sgl_fused_ops.py:102-111).

    A [..., H, D] view such as the K slice of the packed qkv is read in place
    (the reference copies it with .contiguous() first, :108); the result is a
    new contiguous tensor of x's shape, bit-identical to the rmsnorm op on the
    copy (same kernel, same summation order)."""
    assert x.dtype == torch.bfloat16, f"rmsnorm_qk_bf16 needs bf16, got {x.dtype}"
    return _rmsnorm_last(x, _bf16(weight), eps, 0)


def rms_norm_module(x: torch.Tensor, weight: Optional[torch.Tensor] = None,
                    eps: float = 1e-6) -> torch.Tensor:
    """The torch RMSNorm module's forward (dit.py:244-249):
    (x.float() * rsqrt(mean(x.float()^2) + eps)).type_as(x), times weight
    (a separately rounded product) when the module is affine. x: [..., D]
    (the text stream's q or k view, [B, Lt, H, D] inside the packed qkv);
    weight: [D] in x's dtype or None. Returns a new contiguous tensor."""
    D = x.shape[-1]
    if weight is None:
        weight = torch.ones(D, dtype=x.dtype, device=x.device)
    if weight.dtype != x.dtype:
        raise RuntimeError(f"rms_norm_module: weight dtype {weight.dtype} != x dtype {x.dtype}")
    return _rmsnorm_last(x, weight, eps, 1)


def fused_add_gate(residual: torch.Tensor, x: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    """residual + x * gate[:, None] (sgl_fused_ops.py:114-117), a torch op as in the reference."""
    return torch.addcmul(residual, x, gate.unsqueeze(1))


# ---------------------------------------------------------------------------
# Fused forms for callers that can use them.
# ---------------------------------------------------------------------------
def fused_add_gate_layernorm_modulate(
    residual: torch.Tensor,
    x: torch.Tensor,
    gate: torch.Tensor,
    shift: torch.Tensor,
    scale: torch.Tensor,
    *,
    weight: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """(residual', modulated) with residual' = residual + x * gate[:, None] and
    modulated = fused_layernorm_modulate(residual', shift, scale) — the pair of
    calls at dit.py:447-457 in one pass. residual [B, L, D] is updated in place
    (it must be contiguous in its rows) and returned; gate/shift/scale [B, D]."""
    B, L, D = x.shape
    if not residual.is_contiguous():
        raise RuntimeError("residual must be contiguous (it is updated in place)")
    out = fused_add_layernorm_scale_shift(x.reshape(B * L, D), residual.view(B * L, D),
                                          _mod_per_sample(scale, B, L, D),
                                          _mod_per_sample(shift, B, L, D),
                                          gate=_mod_per_sample(gate, B, L, D), gamma=weight,
                                          beta=bias, eps=eps)
    return residual, out.reshape(B, L, D)


def fused_qk_norm_rope_3d_grid_views(
    q: torch.Tensor,
    k: torch.Tensor,
    q_norm_weight: torch.Tensor,
    k_norm_weight: torch.Tensor,
    *,
    grid_hw: Tuple[int, int],
    t0: int,
    rope_dims: Sequence[int],
    theta: float,
    source_id: float = 0.0,
    source_theta: float = 256.0,
    source_dim: int = 128,
    eps: float = 1e-6,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """In-place RMSNorm + RoPE of q, k [B, L, H, D] that may be strided views of
    a packed qkv [B, L, 3, H, D] (heads contiguous per token). Angles come from
    the grid position (frame f of L / (H_grid * W_grid) at t0 + f), with the
    optional source-id rotation over the first min(source_dim, D) dims (the
    model's source_id_rope_dim = 128 and source_id_rope_theta = 256,
    dit.py:549-550,792), exactly as Transformer3DModel builds its tables
    (dit.py:745-809, 918-933); no tables are read. Returns (q, k)."""
    if q.dtype != torch.bfloat16 or k.dtype != torch.bfloat16:
        raise RuntimeError("q/k must be bf16")
    B, L, H, D = q.shape
    if q.stride(-1) != 1 or q.stride(-2) != D or k.stride(-1) != 1 or k.stride(-2) != D:
        raise RuntimeError("heads of a token must be contiguous in q and k")
    freqs = rope_freqs(D, rope_dims, theta, source_theta, source_dim)
    qw = q_norm_weight.to(torch.bfloat16).contiguous()
    kw = k_norm_weight.to(torch.bfloat16).contiguous()
    fused_qk_norm_rope_3d_grid(q, k, L, H, eps, qw, kw, freqs, rope_dims, grid_hw, t0, source_id)
    return q, k


def quantize_activation_fp8(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """The activation side of Fp8Linear.forward (fp8_linear.py:140-144, 166):
    x [..., K] -> (x_q fp8 e4m3fn [M, K], x_scale fp32 [M, 1]) with M = numel / K."""
    return _quantize_activation(x)


def gelu_quantize_activation_fp8(h: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """quantize_activation_fp8(torch.nn.functional.gelu(h, approximate="tanh")) in
    one pass (the MLP activation of dit.py:433 and the activation side of the
    next Fp8Linear.forward, fp8_linear.py:140-166): h [..., K] bf16/fp16 ->
    (x_q fp8 e4m3fn [M, K], x_scale fp32 [M, 1]). The activation is evaluated
    in fp32 and rounded to h's dtype before it is quantized, as the two calls do."""
    return _gelu_quantize_activation(h)


def _mod_per_sample(t: torch.Tensor, B: int, L: int, D: int) -> torch.Tensor:
    """A modulation vector as the fused norm ops take it, without copies: [B, D]
    or [B, 1, D] -> [B, D] (one row per sample of L rows; [D] when B == 1),
    [B, L, D] -> [B*L, D] (a row per token)."""
    if t.numel() == B * D:
        return t.reshape(D) if B == 1 else t.reshape(B, D)
    return t.reshape(B * L, D)


def layernorm_modulate_fp8(
    x: torch.Tensor,
    shift: torch.Tensor,
    scale: torch.Tensor,
    *,
    weight: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """quantize_activation_fp8(fused_layernorm_modulate(x, shift, scale)) in one
    pass: x [B, L, D], shift/scale [B, D], [B, 1, D] or [B, L, D] ->
    (x_q [B*L, D], x_scale [B*L, 1]), byte-identical to the two calls."""
    return _add_gate_layernorm_modulate_fp8(x, None, None, weight, bias, scale, shift, eps)


def fused_add_gate_layernorm_modulate_fp8(
    residual: torch.Tensor,
    x: torch.Tensor,
    gate: torch.Tensor,
    shift: torch.Tensor,
    scale: torch.Tensor,
    *,
    weight: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """fused_add_gate_layernorm_modulate followed by quantize_activation_fp8 of
    its modulated output, in one pass: returns (residual', x_q [B*L, D],
    x_scale [B*L, 1]); residual [B, L, D] is updated in place."""
    if not residual.is_contiguous():
        raise RuntimeError("residual must be contiguous (it is updated in place)")
    x_q, x_scale = _add_gate_layernorm_modulate_fp8(x, residual, gate, weight, bias, scale, shift,
                                                    eps)
    return residual, x_q, x_scale


def commit_kv_pool(pool_k: torch.Tensor, pool_v: torch.Tensor, stage_k: torch.Tensor,
                   stage_v: torch.Tensor, offset: int, commit_cos: torch.Tensor,
                   commit_sin: torch.Tensor) -> None:
    """The graph runner's commit (graph_runner.py:137-142): for every layer li,
    pool_k[li, :, offset:offset+T] = apply_rotary_emb(stage_k[li], (cos, sin)) and
    pool_v[li, :, offset:offset+T] = stage_v[li], as one launch instead of one
    RoPE and two copies per layer. pool_*: [L, B, P, H, D]; stage_*: [L, B, T, H, D];
    commit_cos/sin: fp32 [1, T, D]. Bit-identical to the loop."""
    kv_commit_rope(stage_k, pool_k, offset, commit_cos, commit_sin, src_v=stage_v, dst_v=pool_v)


FP8_MAX = 448.0


def quantize_weight_per_channel(w: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Fp8Linear's weight preparation (fp8_linear.py:100-110, the path without
    fast accumulation): w [N, K] -> (w_q fp8 [K, N] column-major, scale fp32 [N])
    with scale = max|w[n, :]| / 448 (floored at 1e-8 / 448)."""
    w_kn = w.to(torch.bfloat16).t().contiguous()
    absmax = w_kn.abs().amax(dim=0).to(torch.float32).clamp_min(1e-8)
    scale = absmax / FP8_MAX
    w_q_rm = (w_kn.float() / scale.unsqueeze(0)).clamp(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn)
    return w_q_rm.t().contiguous().t(), scale


def fp8_linear(x: torch.Tensor, weight_fp8: torch.Tensor, weight_scale: torch.Tensor,
               bias: Optional[torch.Tensor] = None, out_dtype=torch.bfloat16) -> torch.Tensor:
    """Fp8Linear.forward (fp8_linear.py:155-169): x [..., K] bf16 -> per-token
    fp8 + scales -> fp8_scaled_mm with the per-channel weight scales and bias."""
    if x.requires_grad:
        x = x.detach()  # its quantized form carries no gradient
    return _fp8_linear(x, weight_fp8, weight_scale, bias, out_dtype)


def fp8_linear_quantized(x_q: torch.Tensor, x_scale: torch.Tensor, weight_fp8: torch.Tensor,
                         weight_scale: torch.Tensor, bias: Optional[torch.Tensor] = None,
                         out_dtype=torch.bfloat16) -> torch.Tensor:
    """The GEMM half of fp8_linear for activations already quantized in a norm's
    epilogue (layernorm_modulate_fp8 / fused_add_gate_layernorm_modulate_fp8)."""
    return fp8_scaled_mm(x_q, weight_fp8, x_scale, weight_scale, out_dtype, bias)
