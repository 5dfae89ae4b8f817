"""The FP8 GEMM's streaming kernel (up to 80 rows, chosen by the default launch shape): every
count of 16-row blocks, exact and one row over, with the column blocks that the width
selects (narrow, 4096, 12288 columns and ragged), whole and partial 128-byte steps of K,
fewer and more steps than the eight waves that share them;
NaN padding around the operands. Bar: test_gpu_fp8_gemm's; the same bits on every run."""
from __future__ import annotations

import pytest
import torch

from test_gpu_fp8_gemm import check, operands
from test_gpu_gemm_ktail import _padded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81])
@pytest.mark.parametrize("N,K,dtype", [(8, 16, torch.bfloat16), (24, 1168, torch.float16),
                                       (4096, 256, torch.bfloat16), (4104, 1040, torch.bfloat16),
                                       (8200, 512, torch.float16), (12288, 128, torch.bfloat16),
                                       (16376, 1152, torch.bfloat16)])
def test_few_rows(dev, M, N, K, dtype):
    import joyomni_ops as jo
    a, w, sa, sb, bias = operands(M, N, K, M + N + K, dtype, with_bias=M % 2 == 1)
    ad = _padded(a, 16).to(dev).view(torch.float8_e4m3fn)[:, :K]
    wd = _padded(w, 48).to(dev).view(torch.float8_e4m3fn)[:, :K]
    call = lambda: jo.fp8_scaled_mm(ad, wd.t(), sa.to(dev), sb.to(dev), dtype,  # noqa: E731
                                    bias.to(dev) if bias is not None else None)
    out = call()
    check(out, a, w.t(), sa, sb, bias, f"[{M},{N},{K}]")
    assert torch.equal(out, call())

