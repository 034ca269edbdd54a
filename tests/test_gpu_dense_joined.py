"""Two linears joined to the fp32 stream in one product, against 64 bits."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# 64 x 64 tiles, 64 x 128, 256 x 256; the last row and column tile of some; K of one tile, of fewer than the stages, of many
@pytest.mark.parametrize("M,N,Ka,Kb,taken", [(1025, 516, 64, 64, True), (1100, 1024, 1024, 2816, True), (1101, 2048, 64, 640, True), (2000, 2048, 128, 64, True), (6000, 2044, 64, 1024, True), (8192, 2048, 192, 64, True),
                                             (8191, 2048, 2048, 5632, True), (1000, 1024, 1024, 2816, False), (17, 256, 64, 64, False), (16, 256, 64, 64, False), (1100, 1024, 96, 64, False),
                                             (1100, 1023, 64, 64, False)])
def test_joined(M, N, Ka, Kb, taken):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    a, b = r(M, Ka + 8)[:, :Ka].bfloat16(), r(M, Kb).bfloat16()                 # rows of a wider buffer
    a = torch.cat([a, a[:, :8]], 1)[:, :Ka]
    wa, wb = (r(N, Ka) * Ka ** -0.5).bfloat16(), (r(N, Kb) * Kb ** -0.5).bfloat16()
    buf = torch.full((M * N + 128,), 5.0, device=DEV)
    x = buf[64:64 + M * N].view(M, N)
    x.copy_(r(M, N))
    x0 = x.clone()
    assert hops.dense_joined(x, 0.3, a, wa, b, wb) is taken
    assert bool((buf[:64] == 5.0).all()) and bool((buf[64 + M * N:] == 5.0).all())
    if not taken:
        assert torch.equal(x, x0)
        return
    y = x0.double() + 0.3 * (a.double() @ wa.double().t() + b.double() @ wb.double().t())
    mag = x0.double().abs() + 0.3 * (a.double().abs() @ wa.double().abs().t() + b.double().abs() @ wb.double().abs().t())
    # fp32 sums of Ka + Kb terms of either sign and the sum with the stream: 2^-18 of the terms' magnitudes
    assert bool(((x.double() - y).abs() <= 2.0 ** -18 * mag).all())


def test_joined_takes_no_other_types():
    x = torch.randn(2000, 256, device=DEV)
    a, w = torch.randn(2000, 64, device=DEV), torch.randn(256, 64, device=DEV)
    assert not hops.dense_joined(x, 1.0, a, w, a, w)
