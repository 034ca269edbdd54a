"""The bf16 dense linear at the edges of its tile shapes: remainders of rows, outputs and K in every tile size, strided inputs, unaligned outputs, every epilogue, groups
with a row gather -- against a 64-bit product.  Bound: half a spacing of the output type (bf16: 2^-8 of the value, fp32: 2^-24) plus fp32 sums of K products,
K 2^-24 sum |x w| at the very worst, 2^-17 here (K <= 5632)."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rand(g, *shape, k=1.0):
    return (torch.randn(*shape, device=DEV, generator=g) * k).bfloat16()


# rows x outputs x K: 64 x 64 tiles, 64 x 128 in two and in three stages, 128 x 128, 256 x 256 (test_tile_shapes.py holds the list to that); K below, at and between the K tiles
# of 32 and 64, and an even and an odd count of them with a remainder
SHAPES = [(17, 8, 8), (63, 24, 40), (65, 130, 64), (129, 200, 72), (300, 1000, 32), (700, 2050, 200), (1537, 1028, 96), (2300, 4100, 136), (4700, 4360, 104), (513, 12, 2056),
          (5000, 5000, 24), (1537, 2172, 1032), (2304, 1028, 520), (6000, 1024, 264), (4700, 4360, 200), (6145, 1400, 1032), (6148, 4032, 232), (8190, 2044, 2056), (8190, 2044, 2088)]


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_dense_tiles(M, N, K, f32):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    wide = _rand(g, M, K + 24)
    x, w, bias = wide[:, 8:8 + K], _rand(g, N, K, k=K ** -0.5), _rand(g, N, k=0.1)          # rows at a stride, first column 16 bytes in
    y = hops.dense_linear(x, w, bias, out_dtype=torch.float32 if f32 else None)
    ref = x.double() @ w.double().t() + bias.double()
    mag = x.double().abs() @ w.double().abs().t() + bias.double().abs()
    bound = (2.0 ** -24 if f32 else 2.0 ** -8) * 1.01 * ref.abs() + 2.0 ** -17 * mag
    assert float(((y.double() - ref).abs() / bound).max()) <= 1.0
    # a row's result depends on its own input only, whatever tile it lies in
    for r in (0, M // 2, M - 1):
        lo = max(0, min(r, M - 17))
        assert torch.equal(hops.dense_linear(x[lo:lo + 17], w, bias, out_dtype=torch.float32 if f32 else None)[r - lo], y[r])


GATED = [(65, 64, 40), (700, 1344, 72), (2300, 4160, 136), (4700, 4416, 104), (1537, 2176, 1032), (4700, 4352, 200), (8190, 2048, 2056)]


@pytest.mark.parametrize("act", [hops.ACT_RELU, hops.ACT_SILU, hops.ACT_GELU_TANH])
@pytest.mark.parametrize("M,N,K", GATED)
def test_dense_tiles_gated(M, N, K, act):
    g = torch.Generator(device=DEV).manual_seed(M + N + K + act)
    gate, up, x = _rand(g, N // 2, K, k=K ** -0.5), _rand(g, N // 2, K, k=K ** -0.5), _rand(g, M, K)
    y = hops.dense_linear(x, hops.group_gate_up(gate, up), gated=True, act=act).double()
    a, u = x.double() @ gate.double().t(), x.double() @ up.double().t()
    f = {hops.ACT_RELU: torch.relu, hops.ACT_SILU: torch.nn.functional.silu, hops.ACT_GELU_TANH: lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[act]
    ref = f(a) * u
    assert float(((y - ref).abs() / (2.0 ** -8 * 1.01 * ref.abs() + 2.0 ** -15 * (a.abs() + 1) * (u.abs() + 1))).max()) <= 1.0


def test_dense_tiles_softcap_and_odd_stride_of_the_output():
    g = torch.Generator(device=DEV).manual_seed(5)
    x, w = _rand(g, 2300, 136), _rand(g, 4101, 136)
    out = torch.full((2300, 4107), 7.0, device=DEV)
    hops.dense_linear(x, w, out_dtype=torch.float32, softcap=30.0, out=out[:, 1:4102])
    ref = 30.0 * torch.tanh((x.double() @ w.double().t()) / 30.0)
    assert torch.allclose(out[:, 1:4102].double(), ref, atol=2e-4, rtol=1e-5)
    assert torch.all(out[:, 0] == 7.0) and torch.all(out[:, 4102:] == 7.0)


@pytest.mark.parametrize("rows", [[0, 70, 1, 64, 129, 0, 36], [300, 0, 0, 500]])
def test_dense_groups_gathered(rows):
    """Rows sorted by group, each reading a gathered row of x; groups without rows."""
    g = torch.Generator(device=DEV).manual_seed(len(rows))
    G, K, N, T = len(rows), 104, 200, 90
    total = sum(rows)
    x, w = _rand(g, T, K), _rand(g, G, N, K, k=K ** -0.5)
    gather = torch.randint(0, T, (total,), device=DEV, generator=g, dtype=torch.int32)
    offs = torch.tensor([sum(rows[:i]) for i in range(G + 1)], dtype=torch.int32, device=DEV)
    y = hops.dense_grouped(x, w, rows=total, offs=offs, gather=gather, out_dtype=torch.float32)
    for i in range(G):
        a, b = int(offs[i]), int(offs[i + 1])
        ref = x[gather[a:b].long()].double() @ w[i].double().t()
        assert torch.allclose(y[a:b].double(), ref, atol=1e-4, rtol=1e-5)
