"""A row of the bf16 dense linear between 2 and 16 rows: the same bits however many rows there are (8 and 16 outputs per block, two waves' sums in one product or not), for deep and shallow K, K that is
no multiple of a wave's step, outputs that are no multiple of a block's, gated pairs and groups."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _same(make):
    y = make(16)
    for M in (2, 3, 7, 8, 9, 15):
        assert torch.equal(make(M), y[:M]), M


@pytest.mark.parametrize("N,K", [(2048, 5632), (2048, 2048), (1024, 1000), (20, 192), (9, 136), (100, 1544), (2052, 2048), (16, 72), (600, 1024), (300, 4104)])
def test_plain(N, K):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x, w = torch.randn(16, K, device=DEV, generator=g).bfloat16(), (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    _same(lambda M: hops.dense_linear(x[:M], w, out_dtype=torch.float32))


@pytest.mark.parametrize("I,K", [(32, 128), (96, 1000), (1408, 1024), (2048, 2056)])
def test_gated(I, K):
    g = torch.Generator(device=DEV).manual_seed(I + K)
    x = torch.randn(16, K, device=DEV, generator=g).bfloat16()
    w = hops.group_gate_up(*((torch.randn(I, K, device=DEV, generator=g) * K ** -0.5).bfloat16() for _ in range(2)))
    _same(lambda M: hops.dense_linear(x[:M], w, gated=True, act=hops.ACT_SILU, out_dtype=torch.float32))


def test_groups():
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w = torch.randn(16, 3 * 1536, device=DEV, generator=g).bfloat16(), torch.randn(3, 24, 1536, device=DEV, generator=g).bfloat16()
    _same(lambda M: hops.dense_grouped(x[:M].contiguous(), w, x_step=1536, y_step=24, out_dtype=torch.float32))
