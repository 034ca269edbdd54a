"""Linears of 16-bit weights over up to 64 rows: the block shapes of grids that leave the chip idle and of those that fill it, 1 to 9 chunks of K in flight, whole and ragged tiles.
Bound: exact 16-bit products, fp32 sums of K terms (2^-23 K of the sum of their absolute values), one rounding to the activation type; split sums may be rounded to it once more."""
import pytest
import torch

from rtp_llm_amd import ops, quant

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("K,N", [(64, 16), (128, 48), (896, 1152), (896, 9728), (640, 33 * 16), (1152, 8 * 16), (4864, 896), (1024, 20000), (440, 16384), (312, 17256),
                                 (4864, 1800), (624, 17160), (1184, 8480), (1848, 11208)])
def test_few_rows_of_16_bit_weights(M, K, N, dtype):
    g = torch.Generator(device=DEV).manual_seed(K + N + M)
    x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
    w = (torch.randn(K, N, device=DEV, generator=g) * K ** -0.5).to(dtype)
    bias = torch.randn(N, device=DEV, generator=g).to(dtype)
    y = ops.linear(x, quant.pack_fp16(w), bias)
    ref = x.double() @ w.double() + bias.double()
    off = (x.double().abs() @ w.double().abs() + bias.double().abs()) * K * 2.0 ** -23
    ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert bool(((y.double() - ref).abs() <= off + 2 * ulp * ref.abs() + 2.0 ** -24).all()), float(((y.double() - ref).abs() - off).max())
