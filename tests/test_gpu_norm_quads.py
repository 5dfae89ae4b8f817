"""The fused norms at row lengths that are a multiple of 4 but not of 8 (16-bit types): the
edges of each thread's chunk count (1, 2, 4, 8 and 16 chunks of four over 256 threads) and
lengths on either side of them (the element-wise kernel), through the oracle comparisons of
test_gpu_norms and test_gpu_norm_quant; and rows of a length that is a multiple of 8 whose
stride is only a multiple of 4."""
from __future__ import annotations

import pytest
import torch

import test_gpu_norm_quant as nq
import test_gpu_norms as nn
from helpers import assert_bf16_within_ulp
from oracle import ops

pytestmark = pytest.mark.gpu

LENGTHS = [4, 252, 260, 1020, 1028, 2044, 2052, 4092, 4100, 8188, 8196, 16380, 16388]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", LENGTHS)
@pytest.mark.parametrize("norm,affine", [("layer", "gamma_beta"), ("layer", "none"),
                                         ("rms", "gamma")])
def test_norm_scale_shift(dev, dtype, N, norm, affine):
    nn.test_fused_norm_scale_shift(dev, dtype, 3, N, norm, affine)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", LENGTHS)
@pytest.mark.parametrize("mode", ["plain", "add", "add_gate"])
def test_norm_quant(abi, dev, stream_handle, dtype, N, mode):
    nq.test_norm_quant_matches_unfused_pair(abi, dev, stream_handle, dtype, 3, N, "layer", mode,
                                            True)


@pytest.mark.parametrize("N", [64, 3072])
def test_rows_at_a_stride_of_four(dev, N):
    import joyomni_ops as jo
    M = 37
    g = torch.Generator().manual_seed(N)
    wide = torch.randn(M, N + 4, generator=g).to(torch.bfloat16)
    x, scale, shift = wide[:, :N], 0.2 * wide[:, 4:], wide[:, 4:]
    y = jo.fused_norm_scale_shift(wide.to(dev)[:, :N], None, None, scale.to(dev), wide.to(dev)[:, 4:],
                                  "layer", 1e-6)
    ref = ops.norm_scale_shift_f32(x, None, None, scale, shift, 0, 1e-6)
    assert_bf16_within_ulp(y, ref, ref.abs().amax(1, keepdim=True), what=f"stride N + 4, N = {N}")
