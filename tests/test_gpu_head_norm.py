"""Head norms of several heads a block (129 to 256 channels, and shorter ones from 4096 heads on) and of one, against 64-bit arithmetic.  Error: sums of at most 1024 squares, one reciprocal root and the gate,
a few roundings of 2^-24 each, then one rounding to the activation type."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,H,vdim", [(1, 1, 4), (3, 5, 32), (7, 3, 36), (33, 2, 64), (5, 16, 128), (9, 3, 132), (2, 7, 256), (3, 2, 260), (5, 3, 30), (65, 1, 128), (512, 8, 4), (1024, 4, 32), (585, 7, 36), (1365, 3, 64), (4097, 1, 30), (257, 16, 100), (64, 64, 128)])
@pytest.mark.parametrize("goff,gate_act,per_head", [(None, "silu", False), (4, "silu", True), (3, "sigmoid", False), (8, "sigmoid", True)])
def test_head_norm(rows, H, vdim, goff, gate_act, per_head, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows + vdim)
    n = H * vdim
    o = torch.randn(rows, n, device=DEV, generator=g) * 3
    w = (1 + 0.3 * torch.randn(n if per_head else vdim, device=DEV, generator=g)).to(dtype)
    gate = None if goff is None else torch.randn(rows, n + 12, device=DEV, generator=g)
    y = hops.head_norm(o, H, vdim, w, 1e-5, gate, goff or 0, gate_act=gate_act)
    x = o.double().view(rows, H, vdim)
    ref = x / (x.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * (w.double().view(H, vdim) if per_head else w.double())
    if goff is not None:
        z = gate.double()[:, goff:goff + n].view(rows, H, vdim)
        ref = ref * (torch.sigmoid(z) if gate_act == "sigmoid" else torch.nn.functional.silu(z))
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert y.dtype == dtype and bool(((y.double().view_as(ref) - ref).abs() <= (ulp + 2e-6) * ref.abs() + 1e-30).all())
