"""The FP8 GEMM up to 80 rows under the default launch shape: its streaming kernel at every
number of row and column blocks that the shape selects, rows exact and one over, whole and
partial 128-byte steps of K, fewer and more steps than the eight waves that share them; and
a grid of row counts and widths, whichever kernel each takes (81 rows and the widest columns
a small tile). NaN padding around the operands. Bar: test_gpu_fp8_gemm's; the same bits on
every run."""
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


# (row blocks, column blocks): (N, K) that select them on 256 CUs.
WIDTHS = {
    (1, 1): [(8, 16), (24, 1040)], (1, 2): [(2008, 16), (4104, 1040)],
    (1, 3): [(6008, 16), (8200, 1040)], (1, 4): [(12296, 16), (12296, 1040)],
    (2, 1): [(8, 16), (24, 1040)], (2, 2): [(4104, 16), (4104, 1040)],
    (2, 3): [(8200, 16), (8200, 1040)], (2, 4): [(12296, 16), (12296, 1040)],
    (3, 1): [(8, 16), (24, 1040)], (3, 2): [(4104, 16), (4104, 1040)],
    (3, 3): [(8200, 16), (8200, 1040)],
    (4, 1): [(8, 16), (24, 1040)], (4, 2): [(4104, 16), (4104, 1040)],
    (4, 3): [(8200, 16), (8200, 1040)],
    (5, 1): [(8, 16), (24, 1040)], (5, 2): [(4104, 16), (4104, 1040)],
    (5, 3): [(8200, 16), (8200, 1040)], (5, 4): [(12296, 1040), (12296, 2320)],
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("blocks,N,K", [(b, *nk) for b, v in WIDTHS.items() for nk in v])
def test_every_width(dev, blocks, N, K, exact, dtype):
    import joyomni_ops as jo
    from joyomni_ops import _abi
    mb, nb = blocks
    M = 16 * mb if exact else 16 * mb - 15
    assert _abi.gemm_plan(M, N, K) == (_abi.JO_GEMM_STREAM, 16 * mb, 16 * nb, 1)
    a, w, sa, sb, bias = operands(M, N, K, M + N + K, dtype, with_bias=exact)
    ad = _padded(a, 16).to(dev).view(torch.float8_e4m3fn)[:, :K]
    wd = _padded(w, 48).to(dev).view(torch.float8_e4m3fn)[:, :K]
    call = lambda: jo.fp8_scaled_mm(ad, wd.t(), sa.to(dev), sb.to(dev), dtype,  # noqa: E731
                                    bias.to(dev) if bias is not None else None)
    out = call()
    check(out, a, w.t(), sa, sb, bias, f"[{M},{N},{K}] {mb}x{nb}")
    assert torch.equal(out, call())
