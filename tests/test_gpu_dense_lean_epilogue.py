"""The tile kernels' stores for the common calls against the general ones (outputs that do not lie on 16 bytes take those): the same bits."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _out(M, n, dtype, pad, off):
    """An [M, n] view whose rows are n + pad apart and which starts off elements behind an aligned address, in a buffer of a marked value."""
    buf = torch.full((M * (n + pad) + off + 64,), 7.0, dtype=dtype, device=DEV)
    return buf, buf[off:off + M * (n + pad)].view(M, n + pad)[:, :n]


# every tile shape: 64x64 (few blocks), 64x128 in three and in two stages, 128x128, 256x256 (test_tile_shapes.py holds the lists to that); rows and columns past the last whole tile
SIZES = [(17, 64, 64), (130, 192, 96), (333, 1088, 1024), (1537, 2176, 136), (700, 11264, 256), (2049, 4160, 512), (3001, 11264, 136), (4099, 4160, 264), (8190, 2048, 2056), (4099, 11264, 2048)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("form", ["relu", "silu", "gelu_tanh", "plain", "bias", "odd columns"])
def test_stores(M, N, K, form):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    if form == "odd columns":
        N -= 3
    gated = form in ("relu", "silu", "gelu_tanh")
    x, w = torch.randn(M, K, device=DEV, generator=g).bfloat16(), (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    n, dtype = (N // 2, torch.bfloat16) if gated else (N, torch.float32)
    kw = dict(gated=True, act=hops.ACTIVATIONS[form]) if gated else dict(out_dtype=torch.float32)
    if form == "bias":
        kw["bias"] = torch.randn(N, device=DEV, generator=g).bfloat16()
    got = []
    for pad, off in ((0, 0), (8 - n % 8, 0), (4 + (-n) % 8, 0), (1, 0), (8, 1)):
        buf, out = _out(M, n, dtype, pad, off)
        hops.dense_linear(x, w, out=out, **kw)
        assert int((buf == 7.0).sum()) >= buf.numel() - M * n                   # nothing beside the outputs
        got.append(out.clone())
    assert all(torch.equal(got[0], o) for o in got[1:])
    y = x.double() @ w.double().t()
    if gated:
        v = y.view(M, N // 64, 2, 32)
        act = {"relu": torch.relu, "silu": torch.nn.functional.silu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[form]
        y = (act(v[:, :, 0]) * v[:, :, 1]).reshape(M, n)
    elif form == "bias":
        y = y + kw["bias"].double()
    # fp32 sums of K products (2^-24 a step at most of sums about 1, as 2^-20), the result's rounding
    assert bool(((got[0].double() - y).abs() <= (2.0 ** -7 if gated else 2.0 ** -16) * y.abs() + 2.0 ** -14).all())


# heads of one row block a wave, of two (two or four trips of the loop over rows), of eight in two phases: every tile shape too
HEADS = [(65, 3, 64, 64), (1537, 8, 192, 128), (200, 5, 96, 40), (1537, 3, 96, 512), (2049, 8, 96, 256), (4099, 8, 256, 508), (8190, 2, 1024, 4092)]


@pytest.mark.parametrize("M,H,R,dv", HEADS)
def test_outputs_times_a_gate(M, H, R, dv):
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.randn(M, H * R, device=DEV, generator=g).bfloat16(), (torch.randn(H, dv, R, device=DEV, generator=g) * R ** -0.5).bfloat16()
    z = torch.randn(M, H * dv + 8, device=DEV, generator=g)
    got = []
    for at in (0, 4, 1):                                                        # on 16 bytes, on 16 bytes, not
        gate = torch.zeros_like(z)[:, at:at + H * dv]
        gate.copy_(z[:, :H * dv])
        got.append(hops.dense_grouped(x, w, x_step=R, y_step=dv, mul_sigmoid=gate))
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    y = torch.cat([x.double()[:, h * R:(h + 1) * R] @ w[h].double().t() for h in range(H)], 1) * torch.sigmoid(z[:, :H * dv].double())
    assert bool(((got[0].double() - y).abs() <= 2.0 ** -7 * y.abs() + 2.0 ** -14).all())
