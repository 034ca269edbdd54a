"""The recurrence of a decode step with a linear beside it in the launch: the same bits as the two calls, whether it is one launch or falls back to two."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows per sequence, head (dim, vdim), the linear (N, K, gated), the mode, whether one launch takes it
@pytest.mark.parametrize("counts,dim,vdim,N,K,gated,mode,takes", [
    ([1, 1], 64, 128, 5632, 1024, True, "gla", True),                     # stages of 512, 2 rows
    ([1] * 4, 64, 128, 11264, 2048, True, "hgrn2", True),                 # 4 rows
    ([1] * 8, 64, 128, 11264, 2048, True, "gla", True),                   # 8 rows
    ([1] * 16, 64, 128, 5632, 1024, True, "gla", True),                   # 9 to 16 rows
    ([2, 1, 2], 64, 128, 1536, 1032, False, "gla", False),                # K that no stage fills: without LDS
    ([1] * 5, 64, 128, 128, 264, True, "hgrn2", True),                    # short K, few blocks
    ([1] * 3, 32, 256, 200, 4096, False, "gla", True),                    # stages of 1024; rows past the last block of 8
    ([1] * 3, 30, 100, 192, 1288, True, "gla", True),                     # 8 key rows a thread of an odd head, the last columns of K in a stage of their own
    ([1] * 3, 128, 128, 11264, 2048, True, "gla", False),                 # 16 key rows a thread
    ([1], 64, 128, 512, 512, True, "gla", False),                         # one row
    ([1] * 17, 64, 128, 512, 512, True, "hgrn2", False),                  # past the few
])
@pytest.mark.parametrize("streamed", [False, True])
def test_a_linear_beside_the_recurrence(counts, dim, vdim, N, K, gated, mode, takes, streamed):
    H, T, n = 4, sum(counts), len(counts)
    g = torch.Generator(device=DEV).manual_seed(dim + N)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    hd, hv, rank = H * dim, H * vdim, 16
    proj = r(T, 2 * hd + 2 * hv + rank)
    w2, b2, norm = (r(hd, rank) * 0.25).bfloat16(), r(hd).bfloat16(), (1 + 0.1 * r(vdim)).bfloat16()
    lower, fbias = torch.sigmoid(r(hd)).bfloat16(), r(hd).bfloat16()
    state = r(n + 1, H, dim, vdim)
    start = torch.tensor([sum(counts[:i]) for i in range(n + 1)], dtype=torch.int32, device=DEV)
    slot, first = torch.randperm(n + 1, device=DEV, generator=g)[:n].int(), torch.tensor([3 * (i % 2) for i in range(n)], dtype=torch.int32, device=DEV)
    x, w = r(T, K).bfloat16(), (r(N, K) * K ** -0.5).bfloat16()
    w.streamed = streamed
    lin = dict(x=x, w=w, gated=gated, act=hops.ACT_RELU) if gated else dict(x=x, w=w, out_dtype=torch.float32)
    assert hops.recur_step_takes(dim, vdim, T, w, gated) is takes
    gla = mode == "gla"

    def run(st, **kw):
        return hops.recur_step(hops.SCAN_GLA if gla else hops.SCAN_HGRN2, proj, 0, hd, 2 * hd, 2 * hd + hv if gla else None, (2 * hd + 2 * hv, w2, b2) if gla else None, None,
                               None if gla else lower, None if gla else fbias, 16.0, dim ** -0.5, H, dim, vdim, start, slot, first, st, norm, 1e-5, torch.bfloat16, **kw)

    s0, s1 = state.clone(), state.clone()
    o0, y0 = run(s0), hops.dense_linear(**lin)
    for _ in range(3):
        s1.copy_(state)
        o1, y1 = run(s1, beside=lin)
        assert torch.equal(o0, o1) and torch.equal(y0, y1) and torch.equal(s0, s1)
