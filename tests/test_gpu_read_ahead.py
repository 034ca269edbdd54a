"""Weights read ahead of their use: by the sort of a mixture's (token, choice) pairs and by the blocks that a grouped linear has left over.  Nothing but time may change."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,E,top", [(65, 16, 1), (97, 3, 2), (1537, 16, 4)])
@pytest.mark.parametrize("words", [1, 63, 64, 65, 128 * 1024 * 2 + 5, 26 << 20])   # less than a line, a line, whole blocks of lines and a rest, more than is read
def test_read_ahead(words, T, E, top):
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, 128, generator=g).bfloat16().to(DEV)
    w = (torch.randn(E, 192, 128, generator=g) * 0.1).bfloat16().to(DEV)
    z = torch.randn(T, E, generator=g).to(DEV)
    ahead = torch.ones(words, dtype=torch.bfloat16, device=DEV)
    outs = []
    for a in (None, ahead):
        ids, wts, offs, src, place, tiles = hops.moe_route_sorted(z, E, 1, 1, top, ahead=a)
        y = hops.dense_grouped(x, w, offs=offs, gather=src, tiles=tiles, rows=T * top, ahead=a)
        n = int(tiles[0])
        assert torch.equal(src[place.long().view(-1)].view(T, top), torch.arange(T, device=DEV, dtype=torch.int32)[:, None].expand(T, top))
        outs.append((ids, wts, offs, tiles[:1 + 2 * n], y[place.long().view(-1)]))
    assert all(torch.equal(p, q) for p, q in zip(*outs))
    assert bool((ahead == 1).all())
