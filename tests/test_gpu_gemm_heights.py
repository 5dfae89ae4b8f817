"""The FP8 GEMM at every tile height of its eight-wave kernel (96 to 256 rows in steps of
16), which the default launch shape picks by how many rounds of tiles each needs on the
card's CUs: a row count that only one height covers in a single round of 256 CUs, ragged by
a few rows and columns, one to five K stages of 128 bytes; against the exact float64 result
at the bar of test_gpu_fp8_gemm (one ulp of the output dtype plus 2^-13 of the scaled sum
of |a*b|)."""
from __future__ import annotations

import pytest
import torch

from test_gpu_fp8_gemm import check, operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", range(96, 257, 16))
@pytest.mark.parametrize("K,dtype", [(128, torch.bfloat16), (256, torch.float16),
                                     (640, torch.bfloat16)])
def test_tile_heights(dev, rows, K, dtype):
    import joyomni_ops as jo
    from joyomni_ops import _abi
    M, N = 16 * rows - 5, 4096 - 8
    assert _abi.gemm_plan(M, N, K) == (_abi.JO_GEMM_PAIR, rows, 256, 1)
    a, w, sa, sb, bias = operands(M, N, K, rows + K, dtype)
    out = jo.fp8_scaled_mm(a.to(dev), w.to(dev).t(), sa.to(dev), sb.to(dev), dtype, bias.to(dev))
    # The first tile, the rows around each wave row's and tile's edge, and the ragged last tile.
    pick = sorted({r for t in range(0, M, rows) for r in
                   (t, t + 15, t + 16, t + rows // 2 - 1, t + rows // 2, t + rows - 1) if r < M} |
                  set(range(rows)) | set(range(M - 32, M)))
    idx = torch.tensor(pick)
    check(out[idx.to(dev)], a, w.t(), sa, sb, bias, f"[{M},{N},{K}] {rows}-row tiles", rows=idx)


@pytest.mark.parametrize("M,N,K", [(128, 32776, 1296), (70, 40960, 1408)])
def test_one_row_of_wide_tiles(dev, M, N, K):
    """128x192 tiles: up to 128 rows, a long K and more columns than 128 of them a CU cover."""
    import joyomni_ops as jo
    from joyomni_ops import _abi
    assert _abi.gemm_plan(M, N, K) == (_abi.JO_GEMM_SMALL, 128, 192, 1)
    a, w, sa, sb, bias = operands(M, N, K, M + K)
    out = jo.fp8_scaled_mm(a.to(dev), w.to(dev).t(), sa.to(dev), sb.to(dev), torch.bfloat16,
                           bias.to(dev))
    check(out, a, w.t(), sa, sb, bias, f"[{M},{N},{K}]")
