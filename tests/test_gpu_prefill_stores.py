"""Prompt linears whose results pass through LDS on their way out against the stores from the accumulators, which outputs off 16 bytes take: the same bits, and nothing beside them."""
import pytest
import torch

from rtp_llm_amd import _C, model, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# tiles of 64 x 256, 128 x 256 and 128 x 512 (256 and more columns a block), the last row tile of some rows and the last column tile of some columns; N of 8 but not 16 has no such gated rows
SHAPES = [(1537, 256, 1160), (300, 256, 37888), (1100, 256, 8208), (257, 128, 37896), (1537, 384, 8208), (700, 128, 37880), (4096, 128, 4608), (1537, 512, 37880), (1537, 1024, 8208)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["w4", "int8", "fp16"])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_stores(kind, dtype, M, K, N):
    g = torch.Generator().manual_seed(M + N)
    c = model.synth_linear(K, N, kind, "cpu", g, 128)
    if kind == "fp16":
        c.w = c.w.to(dtype)
    w = c.pack(dtype=dtype).to(DEV)
    x = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    bias = torch.randn(N, generator=g).to(dtype).to(DEV)
    forms = set()
    for epi, b in ((_C.EPI_NONE, None), (_C.EPI_NONE, bias), (_C.EPI_SILU_MUL, bias)):
        n = N // 2 if epi else N
        got = []
        for off in (0, 4):
            buf = torch.full((M * n + 64,), 77.0, dtype=dtype, device=DEV)
            ops.linear(x, w, b, epi, out=buf[off:off + M * n].view(M, n))
            assert bool((buf[:off] == 77.0).all()) and bool((buf[off + M * n:] == 77.0).all())
            got.append(buf[off:off + M * n].clone())
        assert torch.equal(got[0], got[1])


def test_every_tile_with_such_stores_is_among_them():
    lib = _C.lib()
    seen = {lib.mi355_gemm_prefill_form(M, -(-N // 16), -(-K // 128), bf, bits, 128 if bits == 4 else 0, 1) & 15 for M, K, N in SHAPES for bf in (0, 1) for bits in (4, 8, 16)}
    assert {0, 1, 2} <= seen
