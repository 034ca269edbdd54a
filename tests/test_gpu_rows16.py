"""Decode steps of 16-bit weights with norms, rotation, cache write and residual adds inside the linears (up to 8 rows) against the staged launches that 9 rows take: a row's logits, caches and
next token are the same bits, for slices of one to three chunks and of more, one to three tiles of gate_up a block, whole tiles and halves, heads of 64 and 128, activation loads of four and eight rows, 16-bit and INT8 caches."""
import ctypes as C

import pytest
import torch

from oracle import oracle
from rtp_llm_amd import _C, kvcache, model, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CONFIGS = {"deep down": (2, 896, 14, 2, 64, 4864, 2048), "short": (2, 512, 8, 2, 64, 1024, 2048), "heads of 128": (2, 1024, 8, 2, 128, 1536, 2048), "odd chunks": (2, 640, 10, 2, 64, 1920, 2048),
           "whole tiles of qkv": (1, 640, 24, 6, 128, 640, 2048), "two tiles of gate_up": (1, 512, 8, 2, 64, 2560, 2048), "short slice of gate_up": (1, 384, 6, 2, 64, 1152, 2048),
           "both": (1, 256, 4, 2, 64, 3072, 2048), "widest": (1, 1024, 16, 4, 64, 6144, 2048)}


@pytest.mark.parametrize("name", CONFIGS)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kv_int8", [False, True])
def test_same_bits_as_nine_rows(name, dtype, kv_int8):
    cfg = model.ModelConfig(name, *CONFIGS[name], max_pos=512)
    w = model.weights_to(model.synth_model(cfg, "fp16", "cpu", seed=3), DEV)
    page, B = 16, 9
    g = torch.Generator().manual_seed(1)
    table, pos, toks = torch.randperm(4 * B, generator=g).reshape(B, 4).to(torch.int32), torch.randint(0, 61, (B,), generator=g).tolist(), torch.randint(0, cfg.vocab, (B,), generator=g).tolist()

    def run(rows):
        eng = model.DecoderEngine(cfg, w, kv_int8=kv_int8, page=page, num_blocks=4 * B, max_batch=B, max_seq_len=64, device=DEV, dtype=dtype)
        gen = torch.Generator(device=DEV).manual_seed(7)
        for t, s in zip(eng.kv, eng.kv_scale):
            t.copy_(torch.randint(-127, 128, t.shape, device=DEV, generator=gen, dtype=torch.int8) if kv_int8 else torch.randn(t.shape, device=DEV, generator=gen).to(dtype))
            if kv_int8:
                s.fill_(0.01)
        lw = eng._structs[3]
        assert bool(_C.lib().mi355_rows16_ok(rows, *(C.byref(getattr(lw[0], n)) for n in ("qkv", "o", "gate_up", "down")), int(kv_int8), 16)) == (rows <= 8)
        out = []
        eng.set_inputs(toks[:rows], pos[:rows], table[:rows])
        eng.capture(rows)
        for _ in range(3):
            eng.replay(rows, 1)
            torch.cuda.synchronize()
            out.append((eng.logits[:rows].cpu(), eng.token_ids[:rows].cpu()))
        return out, eng

    want, full = run(B)
    for rows in (1, 4, 5, 8):
        got, eng = run(rows)
        for (a, ids), (b, ids_b) in zip(got, want):
            assert torch.equal(a, b[:rows]) and torch.equal(ids, ids_b[:rows]), (rows, float((a - b[:rows]).abs().max()))
        used = table[:rows].flatten().long().to(DEV)
        for l in range(cfg.num_layers):
            assert torch.equal(eng.kv[l][used], full.kv[l][used]) and (not kv_int8 or torch.equal(eng.kv_scale[l][used], full.kv_scale[l][used]))
        assert eng.oob_count() == 0


@pytest.mark.parametrize("hidden,nh,nkv,hd", [(512, 8, 2, 64), (640, 24, 6, 128)], ids=["halves", "whole tiles"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,q_len", [(1, 1), (5, 1), (8, 1), (8, 2), (8, 4), (6, 3)])
def test_cache_write_refuses_as_the_staged_writer(hidden, nh, nkv, hd, dtype, M, q_len):
    """Rotation and cache write in the linear against norm, linear and writer as launches of their own: Q, every byte of the cache and the count of refused rows, with padding rows, positions past
    the pages and past the rotations, block ids past the cache and negative ones, one to four rows a sequence.  Refused: nothing of anybody's page changes."""
    g = torch.Generator().manual_seed(M * 8 + q_len)
    page, max_blocks, nblk, max_pos, N = 8, 4, 40, 27, (nh + 2 * nkv) * hd        # rotations for 27 of the 32 positions that the pages hold
    c = model.synth_linear(hidden, N, "fp16", "cpu", g, 128)
    c.w = c.w.to(dtype)
    w = c.pack(dtype=dtype).to(DEV)
    h, gamma = (torch.randn(M, hidden, generator=g) * 2).to(dtype).to(DEV), (1 + 0.2 * torch.randn(hidden, generator=g)).to(dtype).to(DEV)
    bias, cs = (torch.randn(N, generator=g) * 0.1).to(dtype).to(DEV), oracle.rope_cos_sin(hd, 1e4, max_pos).to(DEV)
    B = M // q_len
    start = torch.randint(0, max_pos - q_len + 1, (B,), generator=g)
    good, table = (start[:, None] + torch.arange(q_len)).reshape(-1).to(torch.int32), torch.randperm(nblk, generator=g)[:B * max_blocks].reshape(B, max_blocks).to(torch.int32)
    cache = torch.randn(kvcache.alloc_layer_cache(nblk, nkv, page, hd, False, "cpu")[0].shape, generator=g).to(dtype)
    lib, ws, st = _C.lib(), ops.weight_struct(w, dtype), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: C.c_void_p(t.data_ptr())

    def both(pos, bt):
        pos, bt, out = pos.to(DEV), bt.to(DEV), []
        for staged in (True, False):
            kv, q, oob = cache.to(DEV), torch.zeros(M, nh, hd, dtype=dtype, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
            layer = ops.kv_struct(kv, None, page, nkv, hd, dtype)
            if staged:
                x, slabs = ops.rmsnorm(h, gamma, 1e-6), torch.empty(16, M, w.N_pad, dtype=torch.float32, device=DEV)
                n = lib.mi355_linear_partial(x.data_ptr(), M, C.byref(ws), slabs.data_ptr(), 16, st)
                assert n >= 1
                rc = lib.mi355_rope_kv_write_rows(None, slabs.data_ptr(), n, w.N_pad, bias.data_ptr(), cs.data_ptr(), hd, max_pos, pos.data_ptr(), bt.data_ptr(), max_blocks, M, q_len, nh,
                                                  C.byref(layer), q.data_ptr(), oob.data_ptr(), st)
            else:
                rc = lib.mi355_rows16_norm_qkv(ptr(h), M, C.byref(ws), ptr(gamma), C.c_float(1e-6), ptr(bias), ptr(cs), max_pos, ptr(pos), ptr(bt), max_blocks, q_len, nh, C.byref(layer), ptr(q),
                                               ptr(oob), None, 16, st)
            assert rc == 0
            torch.cuda.synchronize()
            out.append((q.view(torch.int16).cpu(), kv.view(torch.int16).cpu(), int(oob.item())))
        (q0, kv0, n0), (q1, kv1, n1) = out
        real = pos.cpu() >= 0
        assert torch.equal(q0[real], q1[real]) and torch.equal(kv0, kv1) and n0 == n1
        return kv1, n1

    kv, refused = both(good, table)
    assert refused == 0 and not torch.equal(kv, cache.view(torch.int16))
    for r in {0, M // 2, M - 1}:
        for bad in (-1, max_pos, max_blocks * page, max_blocks * page + 7):        # a row at a time: the others are written as ever
            pos = good.clone()
            pos[r] = bad
            assert both(pos, table)[1] == (bad >= 0)
        for bad in (-1, nblk, nblk + 5):
            bt = table.clone()
            bt[r // q_len, int(good[r]) // page] = bad
            assert both(good, bt)[1] == sum(int(good[i]) // page == int(good[r]) // page for i in range(r // q_len * q_len, r // q_len * q_len + q_len))
    kv, refused = both(torch.full((M,), -1, dtype=torch.int32), table)
    assert refused == 0 and torch.equal(kv, cache.view(torch.int16))
    kv, refused = both(torch.full((M,), max_blocks * page, dtype=torch.int32), table)
    assert refused == M and torch.equal(kv, cache.view(torch.int16))
