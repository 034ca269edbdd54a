"""A shared expert as one more of the grouped linears against the launches of its own, and the sort that gives it its rows."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops, mixers

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T", [1, 64, 65, 128, 1537, 9000])         # whole tiles and a rest, past the pairs of the one-pass sort
@pytest.mark.parametrize("E,top", [(3, 2), (16, 4), (70, 4)])
def test_the_sort_goes_on_over_every_token(T, E, top):
    z = torch.randn(T, E, device=DEV)
    a, b = hops.moe_route_sorted(z, E, 1, 1, top), hops.moe_route_sorted(z, E, 1, 1, top, shared=True)
    n = T * top
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and torch.equal(a[2], b[2][:-1]) and int(b[2][-1]) == n + T
    assert torch.equal(b[3][n:], torch.arange(T, device=DEV, dtype=torch.int32)) and torch.equal(b[3][b[4].flatten().long()], torch.arange(n, device=DEV, dtype=torch.int32) // top)
    na, nb = int(a[5][0]), int(b[5][0])
    assert nb == na + -(-T // 64) and torch.equal(a[5][1:1 + 2 * na], b[5][1:1 + 2 * na])
    assert b[5][1 + 2 * na:1 + 2 * nb].view(-1, 2).tolist() == [[E, n + 64 * m] for m in range(nb - na)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,ff", [(64, 96), (65, 96), (200, 80), (700, 704)])
def test_joint_experts(dtype, T, ff):
    W, E = 256, 8
    g = torch.Generator(device=DEV).manual_seed(T)
    lin = lambda o, i: (torch.randn(o, i, device=DEV, generator=g) * i ** -0.5).to(dtype)
    shared = [lin(ff, W), lin(ff, W), lin(W, ff)]
    own = [[lin(ff, W) for _ in range(E)], [lin(ff, W) for _ in range(E)], [lin(W, ff) for _ in range(E)]]
    build = lambda: mixers.RoutedExperts(mixers.RouterSpec(E, 2), lin(E, W), *own, mixers.GatedMLP(*shared, act="silu"), act="silu")
    h, z = torch.randn(T, W, device=DEV, generator=g).to(dtype), torch.randn(T, E, device=DEV, generator=g)
    one, two = build(), build()
    assert one.joint
    two.joint = False
    assert torch.equal(one.forward(h, z), two.forward(h, z))
    x0 = torch.randn(T, W, device=DEV, generator=g)
    w1 = torch.ones(W, device=DEV, dtype=dtype)
    got = []
    for m in (one, two):
        x = x0.clone()
        got += [x, hops.residual_norm(x, None, m.forward(h, z, defer=True), 1.0, w1, None, 1e-6)[0]]
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])
