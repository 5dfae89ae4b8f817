"""The FP8 GEMM where K is not whole 128-byte stages (any multiple of 16): every remainder
of a stage, with one to five stages, through the eight-wave and the small-tile kernels;
operand rows are padded with NaN codes, so a byte read past K shows, and a NaN inside a row
of either operand reaches exactly its own outputs. Bar: test_gpu_fp8_gemm's."""
from __future__ import annotations

import pytest
import torch

from test_gpu_fp8_gemm import check, operands

pytestmark = pytest.mark.gpu


def _padded(t, pad):
    """t [R, K] fp8 as the leading columns of rows `pad` bytes longer, NaN behind them."""
    R, K = t.shape
    p = torch.full((R, K + pad), 0x7F, dtype=torch.uint8)
    p[:, :K] = t.view(torch.uint8)
    return p


@pytest.mark.parametrize("K", [16, 112, 128 + 16, 128 + 64, 256 + 48, 512 + 80, 512 + 96])
@pytest.mark.parametrize("M,N,shape", [(300, 264, -1), (37, 1000, -1), (700, 4104, -1),
                                       (225, 520, 0), (225, 520, 1), (225, 520, 9), (225, 520, 5),
                                       (225, 520, 6), (225, 520, 8), (225, 520, 10),
                                       (225, 520, 11)])
def test_partial_stage(dev, M, N, K, shape):
    import joyomni_ops as jo
    from joyomni_ops import _abi
    a, w, sa, sb, bias = operands(M, N, K, M + N + K)
    ad = _padded(a, 32).to(dev).view(torch.float8_e4m3fn)[:, :K]
    wd = _padded(w, 64).to(dev).view(torch.float8_e4m3fn)[:, :K]
    _abi.call("jo_set_launch_override", _abi.JO_KNOB_GEMM_SHAPE, shape)
    try:
        out = jo.fp8_scaled_mm(ad, wd.t(), sa.to(dev), sb.to(dev), torch.bfloat16, bias.to(dev))
        check(out, a, w.t(), sa, sb, bias, f"[{M},{N},{K}] shape {shape}")
        # NaN in a row of A (its last 16 bytes) and of B^T (its first byte of the partial stage).
        a2, w2 = ad.clone().view(torch.uint8), wd.clone().view(torch.uint8)
        a2[5, K - 1] = 0x7F
        w2[9, (K - 1) // 128 * 128] = 0x7F
        nan = torch.isnan(jo.fp8_scaled_mm(a2.view(torch.float8_e4m3fn),
                                           w2.view(torch.float8_e4m3fn).t(), sa.to(dev),
                                           sb.to(dev), torch.bfloat16, bias.to(dev))).cpu()
    finally:
        _abi.call("jo_set_launch_override", _abi.JO_KNOB_GEMM_SHAPE, -1)
    want = torch.zeros(M, N, dtype=torch.bool)
    want[5] = True
    want[:, 9] = True
    assert torch.equal(nan, want)
