"""Prompt rows without padding where the blocks with rows fill the chip (16 rows to a wave over shared keys), and where most sequences of a call have none: sequences of no, one, a few and many rows, behind
cached tokens or not, against 64-bit attention over the same pages.  Bound: the weights are rounded to the activation type (2^-11, bf16 2^-8 of each, at most of the
largest value), the result once more."""
import ctypes as C

import pytest
import torch

from rtp_llm_amd import _C, model, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(nh, nkv, hd, page, dtype, lens, start):
    g = torch.Generator(device=DEV).manual_seed(nh + hd + len(lens))
    B, q_len, T = len(lens), max(lens), sum(lens)
    M = -(-max(n + s for n, s in zip(lens, start)) // page) + 1
    kv = torch.full((B * M, 2, nkv, page, hd), float("nan"), device=DEV, dtype=dtype)
    bt = torch.randperm(B * M, generator=torch.Generator().manual_seed(3)).reshape(B, M).int().to(DEV)
    at = [sum(lens[:b]) for b in range(B + 1)]
    q = torch.randn(T, nh, hd, device=DEV, generator=g).to(dtype)
    ref, pos, big = torch.zeros(T, nh, hd, dtype=torch.float64, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV), 0.0
    for b, n in enumerate(lens):
        if n == 0:
            continue
        L = start[b] + n
        k, v = (torch.randn(nkv, L, hd, device=DEV, generator=g).to(dtype) for _ in range(2))
        full = -(-L // page) * page
        pad = lambda t: torch.cat([t, torch.full((nkv, full - L, hd), float("nan"), device=DEV, dtype=dtype)], 1).view(nkv, full // page, page, hd).transpose(0, 1)
        blocks = bt[b, :full // page].long()
        kv[blocks, 0] = pad(k)
        kv[blocks, 1] = pad(v).transpose(2, 3).reshape(full // page, nkv, page, hd)              # values lie [channel][token]
        p = torch.arange(start[b], L, device=DEV)
        pos[at[b]:at[b + 1]] = p.int()
        kk, vv = (t.double().repeat_interleave(nh // nkv, 0) for t in (k, v))
        s = (q[at[b]:at[b + 1]].double().transpose(0, 1) @ kk.transpose(1, 2).contiguous()) * hd ** -0.5
        s = s.masked_fill(torch.arange(L, device=DEV)[None] > p[:, None], float("-inf"))
        ref[at[b]:at[b + 1]] = (s.softmax(-1) @ vv).transpose(0, 1)
        big = max(big, float(v.double().abs().max()))
    lib, L = _C.lib(), ops.kv_struct(kv, None, page, nkv, hd, dtype)
    out = torch.full((T, nh * hd), 7.0, dtype=dtype, device=DEV)
    ws = torch.empty(lib.mi355_paged_attn_workspace_bytes(T, nh, hd, M * page), dtype=torch.uint8, device=DEV)
    row_start = torch.tensor(at, dtype=torch.int32, device=DEV)
    _C.check(lib.mi355_paged_attn_rows_ragged(q.data_ptr(), C.byref(L), bt.data_ptr(), M, pos.data_ptr(), row_start.data_ptr(), B, q_len, T, nh, hd ** -0.5, M * page,
                                              out.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "attn")
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert bool(((out.view(T, nh, hd).double() - ref).abs() <= u * (ref.abs() + big) + 2.0 ** -12 * big).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,page", [(28, 4, 128, 16), (14, 2, 64, 64), (8, 8, 128, 24), (8, 2, 64, 16), (10, 2, 128, 40)])
def test_many_rows(nh, nkv, hd, page, dtype):
    lens = [300, 1, 0, 17, 16, 0, 255, 2, 129, 33] * 10                      # 753 rows in ten sequences, ten times: enough waves with rows for every grouping of heads
    _check(nh, nkv, hd, page, dtype, lens, [(7 * i) % 90 if i % 3 else 0 for i in range(len(lens))])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,page", [(28, 4, 128, 16), (14, 2, 64, 64)])
@pytest.mark.parametrize("lens,start", [([0] * 15 + [64], [0] * 15 + [2048]), ([64] + [0] * 31, [700] * 32), ([1] * 40 + [40], [300] * 41), ([0, 500, 0], [0, 20, 0])])
def test_few_sequences_with_rows(nh, nkv, hd, page, dtype, lens, start):
    _check(nh, nkv, hd, page, dtype, lens, start)


@pytest.mark.parametrize("nh,nkv,hd", [(8, 8, 128), (8, 2, 64), (6, 2, 64)])
@pytest.mark.parametrize("q_len", [16, 33])
def test_many_short_portions(nh, nkv, hd, q_len):
    """Blocks of which some waves have no rows."""
    B = 40960 // (nh * q_len) + 1                                             # rows for 310 blocks' waves and more
    _check(nh, nkv, hd, 16, torch.float16, [q_len] * B, [40 if i % 2 else 0 for i in range(B)])


def test_prefill_when_most_prompts_have_ended():
    """Chunks in which one, two or all of the prompts are left, the block table's rows taken along; against the prompts one by one (fp16 sums in another order: 2^-9 of the largest logit)."""
    cfg = model.ModelConfig("tiny-ragged", 2, 512, 8, 2, 64, 1024, 2048, max_pos=512)
    eng = model.DecoderEngine(cfg, model.weights_to(model.synth_model(cfg, "w4", "cpu", seed=3, zeros="centered"), DEV), kv_int8=False, page=16, num_blocks=96, max_batch=6,
                              max_seq_len=256, device=DEV)
    g = torch.Generator().manual_seed(2)
    prompts = [torch.randint(0, cfg.vocab, (n,), generator=g).tolist() for n in (3, 200, 32, 64, 64, 31)]
    bt = torch.randperm(96, generator=g).reshape(6, 16).int()
    got = eng.prefill(prompts, bt, chunk=32)
    kv = [t.clone() for t in eng.kv]
    one = torch.cat([eng.prefill([p], bt[b:b + 1], chunk=32) for b, p in enumerate(prompts)])
    assert float((got - one).abs().max()) <= 2.0 ** -9 * float(one.abs().max())
    for a, b in zip(kv, eng.kv):
        assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -8 * float(b.float().abs().max())
