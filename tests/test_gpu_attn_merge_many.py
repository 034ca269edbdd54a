"""Decode attention whose last partition merges, where there are more partitions than one round trip of a block's threads holds: parts split over two and over four waves, one wave each,
counters in cache lines of their own and side by side, rows that see fewer partitions than their neighbours -- against the form with a merge launch: the same sums in another order, rounded to
16 bits once (one spacing)."""
import ctypes as C

import pytest
import torch

from rtp_llm_amd import _C, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
APART = 2


@pytest.mark.parametrize("form", [0, APART])
@pytest.mark.parametrize("int8,dtype", [(False, torch.float16), (True, torch.float16), (False, torch.bfloat16)])
@pytest.mark.parametrize("nh,nkv,hd,q_len", [(14, 2, 64, 1), (2, 2, 64, 1), (8, 8, 128, 1), (8, 8, 128, 3), (28, 4, 128, 1), (28, 4, 128, 4), (12, 3, 128, 1)])
@pytest.mark.parametrize("last,max_seq", [([1024], 1280), ([1151], 2048), ([2047, 1100], 2048), ([2048, -1], 4096), ([4095], 4096), ([8191], 8192)])
def test_more_partitions_than_one_round_trip(nh, nkv, hd, q_len, int8, dtype, form, last, max_seq):
    g = torch.Generator(device=DEV).manual_seed(nh + hd + len(last))
    B, page = len(last), 16
    M = max_seq // page
    kv = torch.randint(-100, 100, (B * M, 2, nkv, page, hd), device=DEV, generator=g).to(torch.int8) if int8 else torch.randn(B * M, 2, nkv, page, hd, device=DEV, generator=g).to(dtype)
    scale = torch.rand(B * M, 2, nkv, page, device=DEV, generator=g) * 0.02 + 0.01 if int8 else None
    bt = torch.randperm(B * M, generator=torch.Generator().manual_seed(3)).reshape(B, M).int().to(DEV)
    pos = torch.tensor([[max(-1, p - 200 * (q_len - 1 - i)) for i in range(q_len)] for p in last], dtype=torch.int32, device=DEV).view(-1)
    q = torch.randn(B * q_len, nh, hd, device=DEV, generator=g).to(dtype)
    ref = ops.paged_attention_rows(q, kv, scale, bt, pos, nkv, page, q_len, max_seq)
    lib = _C.lib()
    vp, i32 = C.c_void_p, C.c_int32
    f = C.CFUNCTYPE(i32, vp, vp, vp, i32, vp, i32, i32, i32, C.c_float, i32, vp, i32, vp, C.c_size_t, vp, vp)(("mi355_paged_attn_step", lib))
    L = ops.kv_struct(kv, scale, page, nkv, hd, dtype)
    ws = torch.full((lib.mi355_paged_attn_workspace_bytes(B * q_len, nh, hd, max_seq),), 255, dtype=torch.uint8, device=DEV)
    step = 32 if form & APART else 1
    done = torch.full((B * q_len * nkv, step), 7, dtype=torch.int32, device=DEV)
    done[:, 0] = 0
    want_done = done.clone()
    spacing = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    for _ in range(3):
        out = torch.full_like(ref, 9.0)
        _C.check(f(q.data_ptr(), C.addressof(L), bt.data_ptr(), M, pos.data_ptr(), B, q_len, nh, hd ** -0.5, max_seq, out.data_ptr(), form, ws.data_ptr(), ws.numel(),
                   done.data_ptr(), torch.cuda.current_stream().cuda_stream), "paged_attn_step")
        assert bool(((out - ref).abs().double() <= spacing * ref.abs().double() + 2.0 ** -24).all()) and torch.equal(done, want_done)


@pytest.mark.parametrize("nh,nkv,hd,q_len,B,ctx,inside", [(28, 4, 128, 1, 2, 1000, True), (28, 4, 128, 2, 2, 1000, False), (28, 4, 128, 4, 6, 136, False), (32, 8, 128, 2, 2, 1000, True),
                                                          (16, 2, 128, 2, 4, 600, False), (9, 1, 128, 1, 2, 600, False), (14, 2, 64, 1, 2, 2000, True), (14, 2, 64, 2, 2, 900, True),
                                                          (14, 2, 64, 2, 2, 2000, False), (16, 1, 64, 1, 2, 900, True), (16, 1, 64, 1, 2, 2000, False), (14, 2, 64, 4, 2, 600, False)])
def test_merged_in_the_block_where_it_has_a_thread_for_every_output(nh, nkv, hd, q_len, B, ctx, inside):
    """Beyond that the merge is a launch of its own: the counters are not looked at (here they hold what no arrival completes), elsewhere they are what decides."""
    g = torch.Generator(device=DEV).manual_seed(nh + q_len)
    page = 16
    M = -(-(ctx + 40) // page)
    kv = torch.randn(B * M, 2, nkv, page, hd, device=DEV, generator=g).half()
    bt = torch.arange(B * M, device=DEV, dtype=torch.int32).reshape(B, M)
    pos = (ctx - q_len + torch.arange(q_len, dtype=torch.int32, device=DEV)).repeat(B)
    q = torch.randn(B * q_len, nh, hd, device=DEV, generator=g).half()
    ref = ops.paged_attention_rows(q, kv, None, bt, pos, nkv, page, q_len, M * page)
    lib = _C.lib()
    vp, i32 = C.c_void_p, C.c_int32
    f = C.CFUNCTYPE(i32, vp, vp, vp, i32, vp, i32, i32, i32, C.c_float, i32, vp, i32, vp, C.c_size_t, vp, vp)(("mi355_paged_attn_step", lib))
    L = ops.kv_struct(kv, None, page, nkv, hd, torch.float16)
    ws = torch.zeros(lib.mi355_paged_attn_workspace_bytes(B * q_len, nh, hd, M * page), dtype=torch.uint8, device=DEV)
    done = torch.full((B * q_len * nkv, 32), 1000, dtype=torch.int32, device=DEV)
    out = torch.full_like(ref, 9.0)
    _C.check(f(q.data_ptr(), C.addressof(L), bt.data_ptr(), M, pos.data_ptr(), B, q_len, nh, hd ** -0.5, M * page, out.data_ptr(), APART, ws.data_ptr(), ws.numel(), done.data_ptr(),
               torch.cuda.current_stream().cuda_stream), "paged_attn_step")
    assert bool((done == 1000).all()) != inside and torch.equal(out, ref) != inside
