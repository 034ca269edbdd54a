"""Rows of ragged chunks back to back (no padding rows): writer and attention against the padded form of the same rows, bit for bit where a sequence has more rows than a
column tile (both forms then run the same instance), and a whole prefill against its prompts one by one."""
import ctypes as C

import pytest
import torch

from rtp_llm_amd import _C, model, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("nh,nkv,hd", [(4, 4, 64), (28, 4, 128), (14, 2, 64), (16, 1, 128)])
@pytest.mark.parametrize("lens,start", [([1, 40, 7], [0, 0, 3]), ([33, 0, 64, 2, 0], [5, 0, 100, 0, 9]), ([0, 17], [0, 250])])
def test_rows_without_padding(nh, nkv, hd, int8, dtype, lens, start):
    g = torch.Generator(device=DEV).manual_seed(hd + nh)
    B, q_len, page, M = len(lens), max(lens), 16, 20
    kv = torch.randint(-100, 100, (B * M, 2, nkv, page, hd), device=DEV, generator=g).to(torch.int8) if int8 else torch.randn(B * M, 2, nkv, page, hd, device=DEV, generator=g).to(dtype)
    scale = torch.rand(B * M, 2, nkv, page, device=DEV, generator=g) * 0.02 + 0.01 if int8 else None
    bt = torch.randperm(B * M, generator=torch.Generator().manual_seed(3)).reshape(B, M).int().to(DEV)
    at = [sum(lens[:b]) for b in range(B + 1)]
    T = at[B]
    qkv = torch.randn(T, (nh + 2 * nkv) * hd, device=DEV, generator=g).to(dtype)
    ang = torch.outer(torch.arange(512).float(), 1e4 ** (-torch.arange(0, hd, 2).float() / hd))
    cs = torch.stack((ang.cos(), ang.sin()), -1).contiguous().to(DEV)
    padded = torch.zeros(B, q_len, qkv.shape[1], dtype=dtype, device=DEV)
    pos_p = torch.full((B, q_len), -1, dtype=torch.int32, device=DEV)
    for b, n in enumerate(lens):
        padded[b, :n] = qkv[at[b]:at[b + 1]]
        pos_p[b, :n] = torch.arange(start[b], start[b] + n)
    kv_p, sc_p = kv.clone(), None if scale is None else scale.clone()
    q_p = ops.rope_kv_write_rows(padded.view(B * q_len, -1), None, cs, pos_p.view(-1), bt, kv_p, sc_p, nh, nkv, hd, page, q_len)
    out_p = ops.paged_attention_rows(q_p, kv_p, sc_p, bt, pos_p.view(-1), nkv, page, q_len, M * page).view(B, q_len, -1)

    pos = torch.cat([pos_p[b, :n] for b, n in enumerate(lens)])
    seq = torch.repeat_interleave(torch.arange(B), torch.tensor(lens)).int().to(DEV)
    row_start = torch.tensor(at, dtype=torch.int32, device=DEV)
    st, lib = torch.cuda.current_stream().cuda_stream, _C.lib()
    L = ops.kv_struct(kv, scale, page, nkv, hd, dtype)
    q = torch.empty(T, nh, hd, dtype=dtype, device=DEV)
    _C.check(lib.mi355_rope_kv_write_rows_ragged(qkv.data_ptr(), None, 0, qkv.shape[1], None, cs.data_ptr(), hd, cs.shape[0], pos.data_ptr(), seq.data_ptr(), bt.data_ptr(), M,
                                                 T, 1, nh, C.byref(L), q.data_ptr(), None, st), "rope")
    out = torch.empty(T, nh * hd, dtype=dtype, device=DEV)
    ws = torch.empty(lib.mi355_paged_attn_workspace_bytes(T, nh, hd, M * page), dtype=torch.uint8, device=DEV)
    _C.check(lib.mi355_paged_attn_rows_ragged(q.data_ptr(), C.byref(L), bt.data_ptr(), M, pos.data_ptr(), row_start.data_ptr(), B, q_len, T, nh, hd ** -0.5, M * page,
                                              out.data_ptr(), ws.data_ptr(), ws.numel(), st), "attn")
    assert torch.equal(kv, kv_p) and (scale is None or torch.equal(scale, sc_p))
    for b, n in enumerate(lens):
        assert torch.equal(q[at[b]:at[b + 1]], q_p.view(B, q_len, nh, hd)[b, :n])
        assert torch.equal(out[at[b]:at[b + 1]], out_p[b, :n])


def test_prefill_of_ragged_prompts_equals_one_by_one():
    """Chunks in which some sequences have ended; row counts on both sides of the few-row GEMM.  fp16 results of sums in another order: 2^-9 of the largest logit."""
    cfg = model.ModelConfig("tiny-ragged", 2, 512, 8, 2, 64, 1024, 2048, max_pos=512)
    eng = model.DecoderEngine(cfg, model.weights_to(model.synth_model(cfg, "w4", "cpu", seed=3, zeros="centered"), DEV), kv_int8=False, page=16, num_blocks=64, max_batch=4,
                              max_seq_len=256, device=DEV)
    g = torch.Generator().manual_seed(2)
    prompts = [torch.randint(0, cfg.vocab, (n,), generator=g).tolist() for n in (1, 200, 64, 90)]
    bt = torch.randperm(64, generator=g).reshape(4, 16).int()
    got = eng.prefill(prompts, bt, chunk=64)
    kv = [t.clone() for t in eng.kv]
    one = torch.cat([eng.prefill([p], bt[b:b + 1], chunk=64) for b, p in enumerate(prompts)])
    assert float((got - one).abs().max()) <= 2.0 ** -9 * float(one.abs().max())
    for a, b in zip(kv, eng.kv):
        assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -8 * float(b.float().abs().max())
