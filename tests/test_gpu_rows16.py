"""Decode steps of 16-bit weights with norms, rotation, cache write and residual adds inside the linears (up to 8 rows) against the staged launches that 9 rows take: a row's logits, caches and
next token are the same bits, for slices of one to three chunks and of more, whole tiles and halves, heads of 64 and 128, activation loads of four and eight rows, 16-bit and INT8 caches."""
import ctypes as C

import pytest
import torch

from rtp_llm_amd import _C, model

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CONFIGS = {"deep down": (2, 896, 14, 2, 64, 4864, 2048), "short": (2, 512, 8, 2, 64, 1024, 2048), "heads of 128": (2, 1024, 8, 2, 128, 1536, 2048), "odd chunks": (2, 640, 10, 2, 64, 1920, 2048),
           "whole tiles of qkv": (1, 640, 24, 6, 128, 640, 2048)}


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
