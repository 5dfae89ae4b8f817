"""QK norm + RoPE from fp32 tables and strided q / k (dit_ops.fused_qk_norm_rope_3d and its
K-stage form): bit for bit what the paired ops give for contiguous copies of q and k and
bf16 copies of the tables' pair values, in every form that the direct route takes, and
unchanged in the forms that it leaves to the copies."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # B, L, H, D: one wave's part of the heads, remainders, every head size
    (1, 1, 1, 64), (1, 3, 5, 64), (2, 7, 24, 128), (1, 33, 32, 128), (1, 5, 3, 256),
    (2, 130, 12, 256), (1, 1560, 32, 128),
]


def _inputs(dev, B, L, H, D, wide, row_pad=0):
    g = torch.Generator().manual_seed(B * 1000 + L * 10 + H + D)
    qkv = torch.randn(B, L, 3, H, D, generator=g).to(torch.bfloat16).to(dev)
    qw, kw = ((1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16).to(dev)
              for _ in range(2))
    ang = 100 * torch.rand(L, D // 2, generator=g)
    tabs = []
    for t in (ang.cos(), ang.sin()):
        t = t.repeat_interleave(2, 1) if wide else t
        t = torch.nn.functional.pad(t, (0, row_pad)).to(dev)
        tabs.append(t[:, : t.shape[1] - row_pad])
    return qkv, qw, kw, tabs[0], tabs[1]


def _general(jo, q, k, qw, kw, cos, sin):
    """The paired op on copies, as the reference's caller prepares them."""
    B, L, H, D = q.shape
    q, k = q.clone(memory_format=torch.contiguous_format), k.clone(
        memory_format=torch.contiguous_format)
    if cos.shape[-1] == D:
        cos, sin = cos[..., ::2], sin[..., ::2]
    jo.fused_qk_norm_rope_3d_paired(q.view(B, L * H, D), k.view(B, L * H, D), L, H, 1e-6, qw, kw,
                                    cos.contiguous().to(torch.bfloat16),
                                    sin.contiguous().to(torch.bfloat16))
    return q, k


@pytest.fixture(scope="module")
def dev():
    return "cuda"


@pytest.mark.parametrize("wide,row_pad", [(True, 0), (False, 0), (True, 4), (False, 8)])
@pytest.mark.parametrize("B,L,H,D", SHAPES)
def test_strided_slices_fp32_tables(dev, B, L, H, D, wide, row_pad):
    import joyomni_ops as jo
    from joyomni_ops import dit_ops
    qkv, qw, kw, cos, sin = _inputs(dev, B, L, H, D, wide, row_pad)
    before = qkv.clone()
    q, k = qkv[:, :, 0], qkv[:, :, 1]
    want = _general(jo, q, k, qw, kw, cos, sin)
    tables = (cos, sin) if row_pad else (cos.unsqueeze(0), sin.unsqueeze(0))
    got = dit_ops.fused_qk_norm_rope_3d(q, k, qw, kw, tables)
    for a, b in zip(got, want):
        assert a.is_contiguous() and torch.equal(a, b)
    if L > 1 or B > 1:
        assert torch.equal(qkv, before)  # strided inputs are left as they are
    qkv.copy_(before)  # (the slices of a single token are contiguous: rotated in place)
    stage_want = dit_ops.rmsnorm_qk_bf16(k, kw)
    sq, sk, stage = dit_ops.fused_qk_norm_rope_3d_kstage(q, k, qw, kw, tables)
    assert torch.equal(stage, stage_want)
    assert torch.equal(sq, want[0]) and torch.equal(sk, want[1])
    assert torch.equal(qkv[:, :, 2], before[:, :, 2])


@pytest.mark.parametrize("form", [
    "direct", "contiguous_q", "contiguous_both", "bf16_tables", "fp16_tables", "row_views",
    "misaligned_tables", "head_strided", "batch_expanded", "mixed_strides", "rank4_tables",
    "one_nan",
])
def test_forms_against_the_general_route(dev, form):
    import joyomni_ops as jo
    from joyomni_ops import dit_ops
    B, L, H, D = 2, 9, 8, 128
    qkv, qw, kw, cos, sin = _inputs(dev, B, L, H, D, True)
    q, k = qkv[:, :, 0], qkv[:, :, 1]
    if form == "contiguous_q":
        q = q.contiguous()
    elif form == "contiguous_both":
        q, k = q.contiguous(), k.contiguous()
    elif form in ("bf16_tables", "fp16_tables"):
        dt = torch.bfloat16 if form == "bf16_tables" else torch.float16
        cos, sin = cos.to(dt), sin.to(dt)
    elif form == "row_views":  # every other table row
        cos, sin = (t.repeat_interleave(2, 0)[::2] for t in (cos, sin))
    elif form == "misaligned_tables":
        cos, sin = (torch.cat([t.new_zeros(1), t.flatten()])[1:].view(L, D) for t in (cos, sin))
    elif form == "head_strided":  # heads of a token are not contiguous
        q, k = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k))
    elif form == "batch_expanded":  # both samples read the same rows
        q, k = q[:1].expand(B, -1, -1, -1), k[:1].expand(B, -1, -1, -1)
    elif form == "mixed_strides":  # q from the packed tensor, k from one with another row length
        k = torch.cat([k, k[:, :, :1]], 2)[:, :, :H]
    elif form == "one_nan":
        q[0, 3, 2, 5] = float("nan")
        cos[4, 6:8] = float("inf")
    want = _general(jo, q, k, qw, kw, cos, sin)
    tables = (cos[None, None], sin[None, None]) if form == "rank4_tables" else (cos, sin)
    got = dit_ops.fused_qk_norm_rope_3d(q, k, qw, kw, tables)
    for a, b in zip(got, want):
        assert a.is_contiguous() and torch.equal(a.view(torch.int16), b.view(torch.int16))
    if form.startswith("contiguous"):
        assert got[0].data_ptr() == q.data_ptr()  # rotated in place, as before


def test_captured_pass_replays(dev):
    from joyomni_ops import dit_ops
    qkv, qw, kw, cos, sin = _inputs(dev, 1, 130, 24, 128, True)
    call = lambda: dit_ops.fused_qk_norm_rope_3d(qkv[:, :, 0], qkv[:, :, 1], qw, kw,  # noqa: E731
                                                 (cos.unsqueeze(0), sin.unsqueeze(0)))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        call()
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out = call()
    torch.cuda.synchronize()
    for seed in range(3):
        g = torch.Generator(device=dev).manual_seed(seed)
        qkv.copy_(torch.randn(qkv.shape, generator=g, device=dev))
        want = call()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))


@pytest.mark.parametrize("form", ["sin_with_a_leading_dim", "sin_squeezed_once_too_often",
                                  "weight_of_rank_2"])
def test_forms_that_the_paired_op_refuses(dev, form):
    """sin loses a leading dim only where cos does, as the reference's caller squeezes them, and
    the weights are 1D."""
    from joyomni_ops import dit_ops
    L = 1 if form == "sin_squeezed_once_too_often" else 5
    qkv, qw, kw, cos, sin = _inputs(dev, 2, L, 4, 64, True)
    if form == "sin_with_a_leading_dim":
        sin = sin.unsqueeze(0)
    elif form == "sin_squeezed_once_too_often":
        cos = cos.unsqueeze(0)
    else:
        qw = qw.unsqueeze(0)
    with pytest.raises(RuntimeError):
        dit_ops.fused_qk_norm_rope_3d(qkv[:, :, 0], qkv[:, :, 1], qw, kw, (cos, sin))


@pytest.mark.parametrize("kstage", [False, True])
@pytest.mark.parametrize("tables", ["host", "bf16_rank4"])
def test_tables_that_are_converted_first(dev, tables, kstage):
    import joyomni_ops as jo
    from joyomni_ops import dit_ops
    qkv, qw, kw, cos, sin = _inputs(dev, 1, 9, 8, 128, True)
    q, k = qkv[:, :, 0], qkv[:, :, 1]
    want = _general(jo, q, k, qw, kw, cos, sin)
    given = ((cos.cpu(), sin.cpu()) if tables == "host" else
             (cos.to(torch.bfloat16)[None, None], sin.to(torch.bfloat16)[None, None]))
    call = dit_ops.fused_qk_norm_rope_3d_kstage if kstage else dit_ops.fused_qk_norm_rope_3d
    got = call(q, k, qw, kw, given)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
