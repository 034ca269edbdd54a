"""Norms of heads of 128 channels in 16-byte pieces against the kernel of 4-byte ones, which rows off 16 bytes take: the same bits."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# just enough heads, the last block of a few, heads of several rows in one; weight shared, by head or none; gates and denominators or none
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,H", [(4096, 1), (4099, 1), (1367, 3), (456, 16)])
@pytest.mark.parametrize("weight,gate_act,over", [(1, "silu", False), (2, "sigmoid", True), (0, None, True)])
def test_same_bits(rows, H, weight, gate_act, over, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows + H)
    n = H * 128
    o = torch.randn(rows, n, device=DEV, generator=g) * 3
    o[0] = 0.0
    o[1, 5] = float("inf")
    wide = torch.zeros(rows, n + 3, device=DEV)
    wide[:, 1:1 + n] = o
    w = (1 + 0.3 * torch.randn(n if weight == 2 else 128, device=DEV, generator=g)).to(dtype) if weight else None
    gate = torch.randn(rows, n + 8, device=DEV, generator=g) if gate_act else None
    den = torch.rand(rows, H, device=DEV, generator=g) + 0.5 if over else None
    a, b = (hops.head_norm(x, H, 128, w, 1e-5, gate, 4 if gate_act else 0, out_dtype=dtype, gate_act=gate_act or "silu", den=den) for x in (o, wide[:, 1:1 + n]))
    assert torch.equal(torch.nan_to_num(a, nan=7.0), torch.nan_to_num(b, nan=7.0)) and bool(a[2:].isfinite().all())
