"""The bf16 dense linear on 2 to 16 rows: 8 and 16 outputs per block on either side of the row, output and K rules, against a 64-bit product.  Bound: half a spacing of the
output (fp32 2^-24, bf16 2^-8 with the activation's slope) plus fp32 sums, 2^-17 sum |x w|."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M", [2, 7, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(8, 128), (9, 64), (20, 192), (100, 200), (200, 2048), (2048, 5632), (3072, 1984), (3090, 128), (16, 72)])
def test_few_rows(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    x, w = torch.randn(M, K + 8, device=DEV, generator=g).bfloat16()[:, :K], (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    bias = torch.randn(N, device=DEV, generator=g).bfloat16()
    y = hops.dense_linear(x, w, bias, out_dtype=torch.float32).double()
    ref = x.double() @ w.double().t() + bias.double()
    mag = x.double().abs() @ w.double().abs().t() + bias.double().abs()
    assert float(((y - ref).abs() / (2.0 ** -24 * 1.01 * ref.abs() + 2.0 ** -17 * mag)).max()) <= 1.0


@pytest.mark.parametrize("M", [2, 8, 9])
@pytest.mark.parametrize("I,K", [(32, 128), (96, 192), (2816, 1024), (3104, 64)])
def test_few_rows_gated(M, I, K):
    g = torch.Generator(device=DEV).manual_seed(M + I)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    gate, up = ((torch.randn(I, K, device=DEV, generator=g) * K ** -0.5).bfloat16() for _ in range(2))
    y = hops.dense_linear(x, hops.group_gate_up(gate, up), gated=True, act=hops.ACT_SILU).double()
    a, u = x.double() @ gate.double().t(), x.double() @ up.double().t()
    ref = torch.nn.functional.silu(a) * u
    assert float(((y - ref).abs() / (2.0 ** -8 * 1.01 * ref.abs() + 2.0 ** -15 * (a.abs() + 1) * (u.abs() + 1))).max()) <= 1.0


def test_few_rows_through_every_group():
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w = torch.randn(5, 3 * 128, device=DEV, generator=g).bfloat16(), torch.randn(3, 24, 128, device=DEV, generator=g).bfloat16()
    y = hops.dense_grouped(x, w, x_step=128, y_step=24, out_dtype=torch.float32).double()
    ref = torch.cat([x[:, i * 128:(i + 1) * 128].double() @ w[i].double().t() for i in range(3)], 1)
    assert float((y - ref).abs().max()) <= 2.0 ** -17 * 128 * 4
