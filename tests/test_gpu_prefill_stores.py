"""Prompt linears whose results pass through LDS on their way out against the stores from the accumulators, which outputs off 16 bytes take: the same bits, and nothing beside them."""
import pytest
import torch

from rtp_llm_amd import _C, model, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

KINDS = [("w4", 128), ("w4", 64), ("w4", 32), ("int8", 0), ("fp16", 0)]

# tiles of 64 x 256, 128 x 256 and 128 x 512 (256 and more columns a block) of each class that has them, in launches of one shape, the last row tile of some rows and the last column tile of some
# columns (test_tile_shapes.py holds the list to that); N of 8 but not 16 has no such gated rows.  A class that takes other tiles for a size, or 128 x 512 in groups of 32, stores from the accumulators
# either way
SHAPES = [(300, 256, 37888), (257, 128, 37896), (1537, 384, 8208), (1537, 512, 37880), (1537, 1024, 8208), (200, 768, 25504), (260, 896, 37472), (389, 896, 29248), (200, 128, 8656), (578, 1024, 29568)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,group", KINDS)
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_stores(M, K, N, kind, group, dtype):
    g = torch.Generator().manual_seed(M + N)
    c = model.synth_linear(K, N, kind, "cpu", g, group or 128)
    if kind == "fp16":
        c.w = c.w.to(dtype)
    w = c.pack(dtype=dtype).to(DEV)
    x = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    bias = torch.randn(N, generator=g).to(dtype).to(DEV)
    for epi, b in ((_C.EPI_NONE, None), (_C.EPI_NONE, bias), (_C.EPI_SILU_MUL, bias)):
        n = N // 2 if epi else N
        got = []
        for off in (0, 4):
            buf = torch.full((M * n + 64,), 77.0, dtype=dtype, device=DEV)
            ops.linear(x, w, b, epi, out=buf[off:off + M * n].view(M, n))
            assert bool((buf[:off] == 77.0).all()) and bool((buf[off + M * n:] == 77.0).all())
            got.append(buf[off:off + M * n].clone())
        assert torch.equal(got[0], got[1])
