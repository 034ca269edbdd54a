"""The GEMM of prefill chunks at the edges of its block shapes: more than 64 rows, remainders of the row, column and K tiles, every operand form, against a
64-bit product with a bound built from the formats: half an ulp of the output, plus 2^-11 sum |x w| where fp16 rounds s (u - z) to the operand (fp16 W4), plus
the fp32 sums (K terms of at most 2^-24 sum |x w|, far from all of one sign: 2^-18)."""
import pytest
import torch

from rtp_llm_amd import _C, model, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _gen(seed):
    return torch.Generator().manual_seed(seed)


def _dense64(c):
    if c.kind == "fp16":
        return c.w.double()
    if c.kind == "int8":
        return c.q.double() * c.scales.double()
    g = c.group_size
    return ((c.q.double().view(-1, g, c.N) - c.z_eff.double()[:, None]) * c.scales.double()[:, None]).view(c.K, c.N)


# every tile shape that a call of its class can take, from 32 x 32 on four K slices (narrow, deep, few rows) to 128 x 512 (many rows, wide; codes under fp16): test_tile_shapes.py
# holds the list to that
SHAPES = [(65, 136, 24), (66, 4864, 64), (129, 1280, 200), (130, 896, 1152), (257, 640, 4096), (513, 384, 9728), (1100, 256, 8208),
          (131, 200, 37880), (201, 136, 37880), (300, 2048, 4104), (1537, 136, 4104), (2050, 136, 24), (517, 384, 37880),
          (257, 136, 37880), (1537, 136, 8208), (257, 136, 8208), (777, 104, 8208),
          (417, 264, 8208), (326, 904, 16392), (263, 1160, 37880), (326, 904, 37880), (130, 520, 16392)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,group", [("w4", 128), ("w4", 64), ("w4", 32), ("int8", 0), ("fp16", 0)])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_prefill_gemm_shapes(kind, group, dtype, M, K, N):
    if group and K % group:
        K = -(-K // group) * group
    c = model.synth_linear(K, N, kind, "cpu", _gen(K + N), group or 128)
    if kind == "fp16":
        c.w = c.w.to(dtype)
    x = (torch.randn(M, K, generator=_gen(M)) * 0.5).to(dtype)
    bias = (torch.randn(N, generator=_gen(3)) * 0.1).to(dtype)
    w = _dense64(c)
    ref = x.double() @ w + bias.double()
    mag = x.double().abs() @ w.abs()
    y = ops.linear(x.to(DEV), c.pack(dtype=dtype).to(DEV), bias.to(DEV)).cpu().double()
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10      # spacing at 1: 8 and 11 significant bits
    bound = ulp / 2 * 1.01 * ref.abs() + (2.0 ** -11 if kind == "w4" and dtype == torch.float16 else 0.0) * mag + 2.0 ** -18 * mag + 1e-6
    over = (y - ref).abs() / bound
    assert float(over.max()) <= 1.0, (float(over.max()), float((y - ref).abs().max()))


# K a multiple of 128 (1 to 9 chunks, odd and even, fewer than the slices of K), every tile shape, the last row tile full, of one row, of some
WHOLE = [(65, 128, 48), (100, 256, 1152), (130, 384, 896), (300, 512, 896), (577, 640, 1152), (129, 1152, 4600), (513, 384, 9728), (640, 1024, 4104), (1100, 256, 8208), (2049, 384, 4104),
         (300, 896, 37880), (1537, 1152, 4104), (150, 384, 37880), (400, 896, 4104), (257, 128, 37880), (1537, 128, 8208), (257, 128, 8208), (187, 128, 37880),
         (325, 768, 37880)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,group", [("w4", 128), ("w4", 64), ("w4", 32), ("int8", 0), ("fp16", 0)])
def test_prefill_gemm_straight_loop(kind, group, dtype):
    """x on 16 bytes (the loop without branches) and off them (the general loop): the same bits."""
    seen = set()
    for M, K, N in WHOLE:
        c = model.synth_linear(K, N, kind, "cpu", _gen(K + N), group or 128)
        if kind == "fp16":
            c.w = c.w.to(dtype)
        w = c.pack(dtype=dtype).to(DEV)
        buf = torch.zeros(M * K + 8, dtype=dtype, device=DEV)
        x = (torch.randn(M, K, generator=_gen(M)) * 0.5).to(dtype).to(DEV)
        off = buf[4:4 + M * K].view(M, K).copy_(x)
        assert x.data_ptr() % 16 == 0 and off.data_ptr() % 16 == 8
        assert torch.equal(ops.linear(x, w).view(torch.int16), ops.linear(off, w).view(torch.int16)), (M, K, N)
        if not _C.lib().mi355_gemm_prefill_rest(M, -(-N // 16), K // 128, int(dtype == torch.bfloat16), w.wbits, group, 1):           # two shapes in one launch: test_gpu_prefill_rest.py
            seen.add(_C.lib().mi355_gemm_prefill_shape(M, -(-N // 16), K // 128, int(dtype == torch.bfloat16), w.wbits))
    can = {0, 1, 2, 3, 4, 5, 6} - ({0} if kind == "fp16" or dtype == torch.bfloat16 else set())
    assert seen >= can, seen


# the shapes of a class that have a loop without branches (any K, x on 16 bytes): the others run the general loop either way
STRAIGHT = {("w4", 128, False): {0, 1, 2, 3}, ("w4", 64, False): {1, 2, 3}, ("w4", 32, False): {1, 3}, ("w4", 128, True): {1}, ("w4", 64, True): {1}, ("w4", 32, True): set(),
            ("int8", 0, False): {0, 1, 2, 3, 4, 5, 6}, ("int8", 0, True): {1, 2, 3, 4, 5, 6}, ("fp16", 0, False): {1, 2, 3, 4, 5, 6}, ("fp16", 0, True): {1, 2, 3, 4, 5, 6}}


@pytest.mark.parametrize("kind,group,bf16", STRAIGHT)
def test_prefill_gemm_both_loops(kind, group, bf16):
    """Calls that take the loop without branches with x on 16 bytes and the general one off them, in every shape that has both: the same bits."""
    dtype, bits = (torch.bfloat16 if bf16 else torch.float16), {"w4": 4, "int8": 8, "fp16": 16}[kind]
    form = lambda M, K, N, whole: _C.lib().mi355_gemm_prefill_form(M, -(-N // 16), K // 128, int(bf16), bits, group, int(whole))
    left = set(STRAIGHT[kind, group, bf16])
    for M, K, N in WHOLE + [(370, 896, 37880), (130, 640, 16392), (580, 384, 11016), (835, 640, 8208), (2000, 896, 4104)]:
        if _C.lib().mi355_gemm_prefill_rest(M, -(-N // 16), K // 128, int(bf16), bits, group, 1):                                     # two shapes in one launch: test_gpu_prefill_rest.py
            continue
        whole, off = form(M, K, N, True), form(M, K, N, False)
        assert off < 16 and (whole >= 16) == (whole & 15 in STRAIGHT[kind, group, bf16])
        if whole & 15 not in left:
            continue
        left.discard(whole & 15)
        c = model.synth_linear(K, N, kind, "cpu", _gen(K + N), group or 128)
        if kind == "fp16":
            c.w = c.w.to(dtype)
        w, x = c.pack(dtype=dtype).to(DEV), (torch.randn(M, K, generator=_gen(M)) * 0.5).to(dtype).to(DEV)
        moved = torch.zeros(M * K + 8, dtype=dtype, device=DEV)[4:4 + M * K].view(M, K).copy_(x)
        assert x.data_ptr() % 16 == 0 and moved.data_ptr() % 16 == 8
        assert torch.equal(ops.linear(x, w).view(torch.int16), ops.linear(moved, w).view(torch.int16)), (M, K, N, whole, off)
    assert not left, left


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["w4", "int8", "fp16"])
def test_prefill_gemm_silu_pairs(kind, dtype):
    """The gate-up epilogue on the same launches, rows independent of how many there are."""
    M, K, I = 195, 896, 608
    c = model.synth_linear(K, 2 * I, kind, "cpu", _gen(5))
    if kind == "fp16":
        c.w = c.w.to(dtype)
    x = (torch.randn(M, K, generator=_gen(6)) * 0.5).to(dtype)
    w = _dense64(c)
    exact, mag = x.double() @ w, x.double().abs() @ w.abs()
    gu = exact.to(dtype).double()
    g, u = gu[:, :I], gu[:, I:]
    act = g / (1 + torch.exp(-g))
    y = ops.linear(x.to(DEV), c.pack(gate_up=True, dtype=dtype).to(DEV), None, _C.EPI_SILU_MUL).cpu().double()
    # what each half of the pair may be off by: the sums' bound of the test above, then one spacing where a sum sits on a rounding boundary; |silu'| <= 1.1
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    off = (2.0 ** -11 if kind == "w4" and dtype == torch.float16 else 0.0) * mag + 2.0 ** -18 * mag + ulp * exact.abs()
    bound = 1.1 * off[:, :I] * (u.abs() + off[:, I:]) + act.abs() * off[:, I:] + ulp * (act * u).abs() + 1e-6
    assert float(((y - act * u).abs() / bound).max()) <= 1.0
