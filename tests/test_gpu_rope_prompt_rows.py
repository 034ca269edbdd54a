"""Rows of prompts through the rotation and into the paged cache, 16 rows a block, against the wave per row and head that tensors off 16 bytes take: the same bits everywhere."""
import pytest
import torch

from rtp_llm_amd import _C, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# the smallest counts of rows that go there and one row less, the last block of a few rows, heads that four does not divide, pages of any size, sequences that start at any row
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,hd,nh,nkv,page", [(206, 128, 28, 4, 16), (205, 128, 28, 4, 16), (64, 64, 14, 2, 64), (1058, 128, 5, 1, 24), (300, 64, 32, 32, 16), (1055, 128, 28, 4, 16), (257, 64, 3, 1, 12)])
def test_same_bits(T, hd, nh, nkv, page, dtype):
    g = torch.Generator().manual_seed(T + hd)
    seqs, blocks = 3, -(-T // page) + 1
    count = seqs * blocks + 2
    row_seq = torch.sort(torch.randint(0, seqs, (T,), generator=g, dtype=torch.int32)).values
    pos, seen = torch.zeros(T, dtype=torch.int32), [3] * seqs
    for t in range(T):
        pos[t] = seen[row_seq[t]]
        seen[row_seq[t]] += 1
    pos[::37] = -1                                                          # padding rows
    pos[5::41] = blocks * page + 7                                          # past the block table
    table = torch.randperm(count, generator=g)[:seqs * blocks].int().view(seqs, blocks)
    table[0, 0] = count + 5                                                 # no such block
    ncol = (nh + 2 * nkv) * hd
    qkv, bias = torch.randn(T, ncol, generator=g).to(dtype).to(DEV), torch.randn(ncol, generator=g).to(dtype).to(DEV)
    qkv[0] = -0.0
    qkv[1, :4] = float("nan")
    qkv[2, :4] = float("inf")
    moved = torch.zeros(T * ncol + 8, dtype=dtype, device=DEV)[4:4 + T * ncol].view(T, ncol).copy_(qkv)
    cs = torch.randn(blocks * page + 8, hd // 2, 2, generator=g).to(DEV)
    pos, row_seq, table = pos.to(DEV), row_seq.to(DEV), table.to(DEV)
    for b in (bias, None):
        got = []
        for x in (moved, qkv):
            kv, oob, q = torch.zeros(count, 2, nkv, page * hd, dtype=dtype, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV), torch.full((T * nh * hd + 64,), 7.0, dtype=dtype, device=DEV)
            layer = ops.kv_struct(kv, None, page, nkv, hd, dtype)
            _C.check(_C.lib().mi355_rope_kv_write_rows_ragged(x.data_ptr(), None, 0, ncol, b.data_ptr() if b is not None else None, cs.data_ptr(), hd, cs.shape[0], pos.data_ptr(), row_seq.data_ptr(),
                                                              table.data_ptr(), blocks, T, 1, nh, _C.C.byref(layer), q.data_ptr(), oob.data_ptr(), torch.cuda.current_stream().cuda_stream))
            got.append((kv.view(torch.int16), q.view(torch.int16), oob))
        assert int(got[0][2]) > 0 and bool((got[0][0] != 0).any())
        assert all(torch.equal(m, n) for m, n in zip(*got))
