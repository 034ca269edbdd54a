"""Prompts in several passes: two of them in flight and one after the other are the same launches, so everything they leave is the same bits."""
import pytest
import torch

from rtp_llm_amd import model

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _OneAtATime:
    """The library as it answers where passes do not overlap (they then share one workspace)."""

    def __init__(self, lib):
        self._lib = lib

    def __getattr__(self, name):
        return (lambda handle, rows: 0) if name == "mi355_decoder_prefill_overlaps" else getattr(self._lib, name)


# one prompt of 2 and of 7 passes, prompts that end in different passes, on top of cached tokens; few rows (decode kernels) and many
@pytest.mark.parametrize("lens,start,chunk", [([40], [0], 32), ([200], [0], 32), ([3, 200, 32, 64, 1, 31], [0] * 6, 32), ([150, 90], [40, 7], 16), ([230, 230], [0, 0], 100)])
@pytest.mark.parametrize("kv_int8,dtype", [(False, torch.float16), (True, torch.bfloat16)])
def test_passes_in_flight_change_nothing(lens, start, chunk, kv_int8, dtype):
    cfg = model.ModelConfig("tiny-passes", 3, 512, 8, 2, 64, 1024, 2048, max_pos=512)
    eng = model.DecoderEngine(cfg, model.weights_to(model.synth_model(cfg, "w4", "cpu", seed=3, zeros="centered"), DEV), kv_int8=kv_int8, page=16, num_blocks=96,
                              max_batch=6, max_seq_len=256, device=DEV, dtype=dtype)
    g = torch.Generator().manual_seed(2)
    prompts = [torch.randint(0, cfg.vocab, (n,), generator=g).tolist() for n in lens]
    bt = torch.randperm(96, generator=g).reshape(6, 16).int()[:len(lens)]
    lib = eng.lib
    runs = []
    for turn in range(4):                                       # the second and fourth: streams, events and workspaces that have been used
        for t in eng.kv + [s for s in eng.kv_scale if s is not None]:
            t.zero_()
        eng.lib = _OneAtATime(lib) if turn == 2 else lib
        logits = eng.prefill(prompts, bt, chunk=chunk, start=start)
        runs.append([logits.clone()] + [t.clone() for t in eng.kv] + [s.clone() for s in eng.kv_scale if s is not None])
    eng.lib = lib
    for other in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(runs[0], other))


def test_logits_held_are_bounded():
    """Prompts that end one after the other: the passes' logits [live sequences, vocab] are not held all together (528 rows here), and every prompt's row is
    that of its own last pass."""
    cfg = model.ModelConfig("tiny-endings", 2, 512, 8, 2, 64, 1024, 4096, max_pos=1024)
    n = 32
    eng = model.DecoderEngine(cfg, model.weights_to(model.synth_model(cfg, "w4", "cpu", seed=3, zeros="centered"), DEV), kv_int8=False, page=16, num_blocks=n * (n + 1),
                              max_batch=n, max_seq_len=16 * (n + 1), device=DEV)
    g = torch.Generator().manual_seed(5)
    prompts = [torch.randint(0, cfg.vocab, (16 * (b + 1),), generator=g).tolist() for b in range(n)]
    bt = torch.arange(n * (n + 1)).reshape(n, n + 1).int()
    eng.prefill(prompts, bt, chunk=16)                          # the workspace
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    logits = eng.prefill(prompts, bt, chunk=16)
    torch.cuda.synchronize()
    one = n * cfg.vocab * 4
    assert torch.cuda.max_memory_allocated() - before <= 6 * one                          # the result, four times as much, tables and integers
    eng.lib = _OneAtATime(eng.lib)
    assert torch.equal(logits, eng.prefill(prompts, bt, chunk=16))
