"""Attention of many rows per sequence (as many sequences as make the blocks fill the chip) against 64-bit attention over the same pages: every grouping of heads, rows that are no multiple of a tile, rows out of position
order, padding rows, rows behind cached tokens, pages of 16 to 64 tokens, garbage behind the context.  Bound: the weights are rounded to the activation type (2^-11, bf16
2^-8 of each, at most of the largest value), the result once more."""
import pytest
import torch

from rtp_llm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _sequences(nh, nkv, q_len):
    """Sequences that make 256 blocks: up to eight heads of a key/value head, and as many 16-row tiles as eight waves leave room for."""
    hw = max(d for d in range(1, 9) if (nh // nkv) % d == 0)
    return -(-256 // (-(-q_len // (16 * (8 // hw))) * (nh // hw)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,page", [(28, 4, 128, 16), (14, 2, 64, 64), (8, 8, 128, 24), (8, 2, 64, 16), (16, 1, 128, 16), (6, 2, 64, 32), (10, 2, 128, 40)])
@pytest.mark.parametrize("q_len,start", [(16, [0]), (33, [0, 5, 70]), (130, [0, 300]), (64, [1000, 0])])
def test_prompt_rows(nh, nkv, hd, page, dtype, q_len, start):
    g = torch.Generator(device=DEV).manual_seed(nh + hd + q_len)
    B = _sequences(nh, nkv, q_len)
    start = [start[b % len(start)] for b in range(B)]
    M = -(-(max(start) + q_len) // page) + 1
    kv = torch.full((B * M, 2, nkv, page, hd), float("nan"), device=DEV, dtype=dtype)
    bt = torch.randperm(B * M, generator=torch.Generator().manual_seed(3)).reshape(B, M).int().to(DEV)
    pos = torch.full((B, q_len), -1, dtype=torch.int32, device=DEV)
    ref = torch.zeros(B, q_len, nh, hd, dtype=torch.float64, device=DEV)
    q = torch.randn(B, q_len, nh, hd, device=DEV, generator=g).to(dtype)
    big = 0.0
    for b in range(B):
        n = q_len if b == 0 else q_len - 3                               # the rest are padding rows
        L = start[b] + n
        k, v = (torch.randn(nkv, L, hd, device=DEV, generator=g).to(dtype) for _ in range(2))
        for t0 in range(0, L, page):
            c = min(page, L - t0)
            blk = int(bt[b, t0 // page])
            kv[blk, 0, :, :c] = k[:, t0:t0 + c]
            kv[blk, 1].view(nkv, hd, page)[:, :, :c] = v[:, t0:t0 + c].transpose(1, 2)
        at = torch.arange(start[b], L, device=DEV)
        if n > 20:
            at[3], at[17] = at[17].clone(), at[3].clone()                # two rows out of order
        pos[b, :n] = at.int()
        kk, vv = (t.double().repeat_interleave(nh // nkv, 0) for t in (k, v))
        s = (q[b, :n].double().transpose(0, 1) @ kk.transpose(1, 2).contiguous()) * hd ** -0.5
        s = s.masked_fill(torch.arange(L, device=DEV)[None] > at[:, None], float("-inf"))
        ref[b, :n] = (s.softmax(-1) @ vv).transpose(0, 1)
        big = max(big, float(v.double().abs().max()))
    out = ops.paged_attention_rows(q.view(B * q_len, nh, hd), kv, None, bt, pos.view(-1), nkv, page, q_len, M * page).view(B, q_len, nh, hd).double()
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert bool(((out - ref).abs() <= u * (ref.abs() + big) + 2.0 ** -12 * big).all()), float((out - ref).abs().max())


def test_long_context():
    """20000 cached tokens in pages of 16, scattered; every sequence reads the same ones."""
    g = torch.Generator(device=DEV).manual_seed(1)
    L, q_len, page, nh, nkv, hd = 20000, 40, 16, 16, 2, 64
    M, B = -(-L // page), _sequences(16, 2, 40)
    kv = torch.randn(M, 2, nkv, page, hd, device=DEV, generator=g).half()
    bt = torch.randperm(M, generator=torch.Generator().manual_seed(3)).reshape(1, M).int().to(DEV)
    pos = torch.arange(L - q_len, L, device=DEV, dtype=torch.int32)
    q = torch.randn(q_len, nh, hd, device=DEV, generator=g).half()
    out = ops.paged_attention_rows(q.repeat(B, 1, 1), kv, None, bt.repeat(B, 1), pos.repeat(B), nkv, page, q_len, M * page).view(B, q_len, nh, hd)
    assert bool((out == out[:1]).all())
    k = kv[bt[0].long(), 0].transpose(0, 1).reshape(nkv, -1, hd).double().repeat_interleave(nh // nkv, 0)
    v = kv[bt[0].long(), 1].view(M, nkv, hd, page).permute(1, 0, 3, 2).reshape(nkv, -1, hd).double().repeat_interleave(nh // nkv, 0)
    s = (q.double().transpose(0, 1) @ k.transpose(1, 2).contiguous()) * hd ** -0.5
    ref = (s.masked_fill(torch.arange(M * page, device=DEV)[None] > pos[:, None], float("-inf")).softmax(-1) @ v).transpose(0, 1)
    assert float((out[0].double() - ref).abs().max()) <= 2.0 ** -11 * float(v.abs().max())
