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


@pytest.mark.parametrize("N,K", [(2048, 1016), (2048, 1024), (2050, 1032), (4096, 1016), (4097, 1016), (8184, 1024), (8200, 1160), (6152, 2056), (6136, 2048), (64, 5640),
                                 (512, 504), (520, 504), (512, 512), (520, 512), (6144, 504), (6144, 1152), (6136, 1152), (6144, 1160), (8192, 1160), (8200, 1160), (8192, 1792), (8192, 1800),
                                 (2048, 2304), (2048, 2312), (12288, 1856), (12280, 1856), (8192, 1856), (8192, 1864), (16400, 1024), (16384, 1792), (1536, 3072), (1544, 3072), (1536, 2320), (2048, 2568), (2056, 2568),
                                 (2056, 2824), (1024, 968), (1024, 976), (8184, 976), (8192, 976), (4880, 1024), (12280, 1024), (12288, 1024), (4096, 1000), (4088, 1000), (8192, 488), (4096, 2040), (4096, 2048), (8184, 2048), (8200, 2048), (4096, 1960), (4096, 2056), (12280, 1048), (12288, 1160)])
def test_few_rows_forms(N, K):
    """Either side of each rule that picks the form (2, 4 and 8 rows; K 512, 1024, 1152, 1792, 1856, 2048, 2304, K that fills the stages and K that leaves a twentieth empty; 512, 4096, 6144, 8192, 12288 weight rows; four chains
    and eight), stages and columns of a stage (256 blocks, columns loaded for nothing, 24 MB), a last stage with one piece: against a 64-bit product, the same bits for any number of rows, alone and in a launch of two."""
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x, w = torch.randn(16, K, device=DEV, generator=g).bfloat16(), (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    x2, w2 = torch.randn(16, 72, device=DEV, generator=g).bfloat16(), torch.randn(64, 72, device=DEV, generator=g).bfloat16()
    y = hops.dense_linear(x, w, out_dtype=torch.float32)
    ref, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert float(((y.double() - ref).abs() / (2.0 ** -24 * 1.01 * ref.abs() + 2.0 ** -17 * mag)).max()) <= 1.0
    gated = hops.dense_linear(x2, w2, gated=True, act=hops.ACT_SILU)
    for M in (2, 3, 4, 5, 8, 9, 16):
        a, b = hops.dense_pair(dict(x=x[:M], w=w, out_dtype=torch.float32), dict(x=x2[:M], w=w2, gated=True, act=hops.ACT_SILU))
        assert torch.equal(hops.dense_linear(x[:M], w, out_dtype=torch.float32), y[:M]) and torch.equal(a, y[:M]) and torch.equal(b, gated[:M]), M
    a, b = hops.dense_pair(dict(x=x2, w=w2, gated=True, act=hops.ACT_SILU), dict(x=x, w=w, out_dtype=torch.float32))
    assert torch.equal(a, gated) and torch.equal(b, y)


@pytest.mark.parametrize("N,K", [(448, 488), (1984, 504), (2048, 504), (1984, 1032), (1984, 1024), (4096, 968), (4032, 968), (2048, 1024), (2048, 1032), (4096, 1160), (8128, 1000), (8192, 976), (12224, 1024), (12288, 1024)])
def test_few_rows_gated_forms(N, K):
    """Gated weights either side of their rules (2048, 4096, 8192, 12288 weight rows; K 1024; K that fills the stages) against 64-bit products, the same bits for any number of rows.  silu(g) u: both sums are off by 2^-17 of
    their magnitudes at most (as above), silu's slope is below 1.1, __expf and the division add a few 2^-24 of the gate."""
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x, w = torch.randn(16, K, device=DEV, generator=g).bfloat16(), (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    y = hops.dense_linear(x, w, gated=True, act=hops.ACT_SILU, out_dtype=torch.float32)
    gate, up = (x.double() @ v.double().t() for v in (w.view(-1, 64, K)[:, :32].reshape(-1, K), w.view(-1, 64, K)[:, 32:].reshape(-1, K)))
    mag_g, mag_u = (2.0 ** -17 * (x.double().abs() @ v.double().abs().t()) for v in (w.view(-1, 64, K)[:, :32].reshape(-1, K), w.view(-1, 64, K)[:, 32:].reshape(-1, K)))
    ref = torch.nn.functional.silu(gate) * up
    assert bool(((y.double() - ref).abs() <= 1.1 * mag_g * (up.abs() + mag_u) + torch.nn.functional.silu(gate).abs() * mag_u + 2.0 ** -20 * ref.abs() + 1e-30).all())
    for M in (2, 3, 4, 5, 8, 9):
        assert torch.equal(hops.dense_linear(x[:M], w, gated=True, act=hops.ACT_SILU, out_dtype=torch.float32), y[:M]), M


@pytest.mark.parametrize("M,ldx", [(3, 1 << 30), (16, 143165608), (9, (1 << 29) + 8)])
def test_few_rows_far_apart(M, ldx):
    """Rows of x whose offsets do not fit 32 bits: the bits of the same rows side by side, alone, in a launch of two and through groups."""
    K, g = 1032, torch.Generator(device=DEV).manual_seed(M)
    flat = torch.empty((M - 1) * ldx + 2 * K, dtype=torch.bfloat16, device=DEV)
    far, x = flat.as_strided((M, 2 * K), (ldx, 1)), torch.randn(M, 2 * K, device=DEV, generator=g).bfloat16()
    far.copy_(x)
    w, wg = (torch.randn(*s, device=DEV, generator=g).bfloat16() * K ** -0.5 for s in ((72, K), (64, K)))
    for a, b in ((x[:, :K], far[:, :K]), (x[:, K:], far[:, K:])):
        for out in (torch.float32, torch.bfloat16):
            assert torch.equal(hops.dense_linear(b, w, out_dtype=out), hops.dense_linear(a, w, out_dtype=out))
        want = [hops.dense_linear(a, wg, gated=True, act=hops.ACT_SILU), hops.dense_linear(a, w)]
        assert all(torch.equal(p, q) for p, q in zip(hops.dense_pair(dict(x=b, w=wg, gated=True, act=hops.ACT_SILU), dict(x=b, w=w)), want))
    w2, gate = torch.stack([w, w.flip(0)]), torch.randn(M, 2 * 72, device=DEV, generator=g)
    run = lambda v: hops.dense_grouped(v, w2, x_step=K, y_step=72, mul_sigmoid=gate)
    assert torch.equal(run(far), run(x))


@pytest.mark.parametrize("N,K", [(6144, 2048), (6136, 2048), (13000, 968), (13008, 968)])
def test_few_rows_streamed(N, K):
    """Weights marked as streamed, on either side of 24 MB: the same bits, alone, in a launch of two and through groups."""
    g = torch.Generator(device=DEV).manual_seed(N)
    w = torch.randn(N, K, device=DEV, generator=g).bfloat16()
    s, small, smalls = w.clone(), w[:64].clone(), w[:64].clone()
    s.streamed = smalls.streamed = True
    for M in (2, 8, 16):
        x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
        y = hops.dense_linear(x, w)
        assert torch.equal(hops.dense_linear(x, s), y)
        for a, b in ((s, smalls), (s, small), (w, smalls)):
            p, q = hops.dense_pair(dict(x=x, w=a), dict(x=x, w=b, gated=True, act=hops.ACT_SILU))
            assert torch.equal(p, y) and torch.equal(q, hops.dense_linear(x, small, gated=True, act=hops.ACT_SILU))
        gs = w[:N // 8 * 8].view(4, N // 8 * 2, K).clone()
        z = hops.dense_grouped(x, gs, y_step=N // 8 * 2)
        gs.streamed = True
        assert torch.equal(hops.dense_grouped(x, gs, y_step=N // 8 * 2), z)
