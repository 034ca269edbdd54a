"""Prompt linears that run two tile shapes in one launch against the general loop in one shape, which x off 16 bytes takes: the same bits, and nothing beside them."""
import math
import random

import pytest
import torch

from rtp_llm_amd import _C, model, ops

DEV = "cuda"

# kind, bf16, M, N, K, (first shape, the rest's, column tiles of the first): last row tiles of some rows in both shapes, a last column tile of some columns, each pair of shapes of each class
CALLS = [("w4", False, 4812, 3416, 1536, (0, 3, 6)), ("w4", False, 9385, 3840, 1024, (0, 1, 6)), ("w4", False, 4627, 3736, 1536, (0, 2, 6)), ("w4", False, 6763, 1192, 1408, (1, 3, 4)),
         ("int8", False, 4119, 3936, 1408, (0, 3, 7)), ("int8", False, 9275, 2056, 1664, (0, 1, 3)), ("int8", False, 6534, 2536, 1664, (0, 2, 4)), ("int8", False, 6982, 1176, 1280, (1, 3, 4)),
         ("w4", True, 6671, 1160, 768, (1, 3, 4)), ("int8", True, 6690, 1176, 1024, (1, 3, 4))]


def rest(kind, bf16, M, N, K, whole=1, group=128):
    bits = 4 if kind == "w4" else 8 if kind == "int8" else 16
    r = _C.lib().mi355_gemm_prefill_rest(M, -(-N // 16), -(-K // 128), int(bf16), bits, group if bits == 4 else 0, whole)
    return (r % 4, r // 4 % 4, r // 16) if r else None


@pytest.mark.gpu
@pytest.mark.parametrize("kind,bf16,M,N,K,pick", CALLS)
def test_same_bits_as_one_shape(kind, bf16, M, N, K, pick):
    assert rest(kind, bf16, M, N, K) == pick and rest(kind, bf16, M, N, K, whole=0) is None
    dtype = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator().manual_seed(M + N)
    w = model.synth_linear(K, N, kind, "cpu", g, 128).pack(dtype=dtype).to(DEV)
    x = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    moved = torch.zeros(M * K + 8, dtype=dtype, device=DEV)[4:4 + M * K].view(M, K).copy_(x)
    bias = torch.randn(N, generator=g).to(dtype).to(DEV)
    for epi, b in ((_C.EPI_NONE, None), (_C.EPI_SILU_MUL, bias)):
        n = N // 2 if epi else N
        got = []
        for a, off in ((moved, 0), (x, 0), (x, 4)):                       # off 4: the stores from the accumulators
            buf = torch.full((M * n + 64,), 77.0, dtype=dtype, device=DEV)
            ops.linear(a, w, b, epi, out=buf[off:off + M * n].view(M, n))
            assert bool((buf[:off] == 77.0).all()) and bool((buf[off + M * n:] == 77.0).all())
            got.append(buf[off:off + M * n].view(torch.int16).clone())
        assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


def _whole_rounds(M, N, first, second, cols):
    """The first shape's tiles end on a round of the chip's 256 places, but for less than a column of them, and leave columns behind; the pair of shapes is one that the launch builds."""
    rows, width = -(-M // 128), 512 if first == 0 else 256
    assert 0 < cols * width < N and -(rows * cols) % 256 < rows and (first, second) in {(0, 1), (0, 2), (0, 3), (1, 3)}


@pytest.mark.parametrize("kind,bf16", [("w4", False), ("w4", True), ("int8", False), ("int8", True)])
def test_first_shape_fills_whole_rounds_and_leaves_some(kind, bf16):
    g, pairs = random.Random(f"{kind} {bf16}"), set()
    sizes = [(M, N, K) for k, b, M, N, K, _ in CALLS if (k, b) == (kind, bf16)]
    sizes += [(int(math.exp(g.uniform(math.log(65), math.log(12000)))), 8 * g.randint(8, 4750), 128 * g.randint(1, 150)) for _ in range(3000)]
    for M, N, K in sizes:
        pick = rest(kind, bf16, M, N, K)
        if pick:
            _whole_rounds(M, N, *pick)
            pairs.add(pick[:2])
            assert rest(kind, bf16, M, N, K, whole=0) is None
    assert pairs == ({(1, 3)} if bf16 else {(0, 1), (0, 2), (0, 3), (1, 3)})
    for k, b, M, N, K, pick in CALLS:
        if (k, b) == (kind, bf16):
            assert rest(k, b, M, N, K) == pick


def test_one_shape_where_two_are_not_built():
    for M in (65, 128, 1000, 4096):                                         # 16-bit weights, groups of 64, fewer blocks than the chip has places for
        assert rest("fp16", True, M, 37888, 3584) is None and rest("w4", False, M, 37888, 3584, group=64) is None
    assert rest("w4", False, 100, 37888, 3584) is None
