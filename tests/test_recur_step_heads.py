"""Which heads the recurrence step of few rows takes (what its launch has an instance for, all other heads walk) and which steps a mixer gives it."""
import types

import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops, mixers


def test_heads_with_an_instance():
    for vdim in range(1, 300):
        for dim in range(1, 300):
            one = vdim % 4 == 0 and vdim <= 256 and dim <= 256 and dim * vdim <= 32768
            fits = one and -(-dim // (256 // (vdim // 4))) <= 36             # key rows of a thread that holds four columns
            assert hops.recur_step_supported(dim, vdim) is fits, (dim, vdim)


# rows of the sequences of a step, whether max_rows says so
@pytest.mark.parametrize("known", [True, False])
@pytest.mark.parametrize("kind,dim,vdim,counts,few", [
    ("gla", 64, 128, [1] * 16, True), ("gla", 64, 128, [2] * 8, True), ("gla", 128, 256, [1, 2], True), ("gla", 64, 128, [3], False), ("gla", 64, 128, [16], False),
    ("gla", 64, 128, [1] * 17, False), ("gla", 184, 176, [1], False), ("hgrn2", 64, 128, [1] * 16, True), ("hgrn2", 64, 128, [2], False), ("hgrn2", 64, 256, [1], True),
    ("hgrn2", 128, 256, [1], False), ("hgrn2", 256, 128, [1], True), ("hgrn2", 64, 128, [8, 8], False)])
def test_steps_of_a_mixer(kind, dim, vdim, counts, few, known):
    H, W = 2, 32
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    w = {n: z(H * c, W) for n, c in (("q", dim), ("k", dim), ("f", dim), ("v", vdim), ("g", vdim))}
    w.update({"a1": z(8, W), "a2": z(H * dim, 8), "a2.b": z(H * dim), "lower": z(H * dim), "f.b": z(H * dim), "norm": z(vdim), "o": z(W, H * vdim)})
    mixer = mixers.GatedLinearRecurrence(mixers.RecurrenceSpec(kind=kind, heads=H, dim=dim, vdim=vdim), w, 1e-5)
    batch = types.SimpleNamespace(max_rows=max(counts) if known else 0, slot=torch.zeros(len(counts), dtype=torch.int32))
    longest = max(counts) if known else sum(counts) - len(counts) + 1                    # unknown: the longest that there may be
    got = mixer.few_rows(sum(counts), batch)
    assert (got is not None) is (few and (known or longest <= (2 if kind == "gla" else 1)))
    assert got is None or got[0].shape[0] == H * (2 * dim + vdim) + (H * vdim + 8 if kind == "gla" else 0)
