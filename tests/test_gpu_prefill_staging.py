"""Activations of the prefill GEMM that the DMA into LDS does not take -- a tensor off 16 bytes -- give the bits of an aligned copy; row counts around the row tiles."""
import pytest
import torch

from rtp_llm_amd import model, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["w4", "int8", "fp16"])
@pytest.mark.parametrize("M,K,N", [(65, 256, 64), (127, 384, 1152), (129, 1152, 4096), (1100, 256, 8208)])
def test_activations_off_16_bytes(kind, dtype, M, K, N):
    c = model.synth_linear(K, N, kind, "cpu", torch.Generator().manual_seed(N), 128)
    if kind == "fp16":
        c.w = c.w.to(dtype)
    w = c.pack(dtype=dtype).to(DEV)
    flat = torch.randn(M * K + 4, generator=torch.Generator().manual_seed(M)).to(dtype).to(DEV)
    off = flat[4:].view(M, K)
    assert off.data_ptr() % 16 == 8
    assert torch.equal(ops.linear(off, w), ops.linear(off.clone(), w))
