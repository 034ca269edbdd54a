"""Launches of steps of few rows: two linears in one (the bits of two calls), and a recurrence with its norm and output gate in one against the same in 64 bits."""
import types

import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops, mixers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# forms of 16 and of 8 outputs a block, 4 and 8 partial sums of K, outputs that end inside a tile, gated and plain; one row and more than 16 rows are two calls
@pytest.mark.parametrize("M", [1, 2, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("K0,N0,K1,N1,gated", [(2048, 6160, 2048, 11264, True), (2048, 2048, 5632, 2048, False), (1024, 528, 1024, 5632, True), (640, 100, 1032, 24, False),
                                               (64, 16, 512, 192, True), (1000, 50, 96, 17000, False)])
def test_pair_is_two_calls(M, K0, N0, K1, N1, gated):
    g = torch.Generator(device=DEV).manual_seed(M + N0)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g).bfloat16()
    a = dict(x=r(M, K0 + 8)[:, :K0], w=r(N0, K0), bias=r(N0), out_dtype=torch.float32)
    b = dict(x=r(M, K1), w=r(N1, K1), gated=gated, act=hops.ACT_SILU if gated else hops.ACT_NONE, out_dtype=torch.bfloat16 if gated else torch.float32)
    for first, second in ((a, b), (b, a)):
        got = hops.dense_pair(first, second)
        for y, d in zip(got, (first, second)):
            assert torch.equal(y, hops.dense_linear(**d))


@pytest.mark.parametrize("mode", ["hgrn2", "gla", "gla-z", "fixed", "fixed-silu"])
@pytest.mark.parametrize("H,dim,vdim,rank", [(16, 64, 128, 16), (3, 32, 64, 4), (2, 128, 256, 16), (2, 256, 128, 24), (5, 40, 96, 3), (1, 7, 4, 1), (4, 100, 100, 8), (1, 144, 208, 8)])
@pytest.mark.parametrize("counts", [[1], [1, 1, 1, 1, 1, 1, 1, 1], [3, 1, 12]])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_recurrence_of_few_rows(mode, H, dim, vdim, rank, counts, dtype):
    """Bound: gates and updates in fp32 over at most 12 tokens leave the state within 2^-18 of its largest value.  An output is a sum over keys of state times query: it is off by 2^-17
    of the sum of their absolute values (state, query, 256 additions), which the norm divides by the head's RMS and the weight and gate multiply; then one rounding to the act type."""
    g = torch.Generator(device=DEV).manual_seed(H * dim + vdim)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T, n, hd, hv = sum(counts), len(counts), H * dim, H * vdim
    start = torch.tensor([sum(counts[:i]) for i in range(n + 1)], dtype=torch.int32, device=DEV)
    slot = torch.randperm(n + 2, generator=torch.Generator().manual_seed(n))[:n].to(DEV, torch.int32)
    first = torch.tensor([5 if i % 2 == 0 else 0 for i in range(n)], dtype=torch.int32, device=DEV)
    proj = r(T, 2 * hd + 2 * hv + rank + 3)[:, :2 * hd + 2 * hv + rank]
    qo, ko, vo, go, ao = 0, hd, 2 * hd, 2 * hd + hv, 2 * hd + 2 * hv
    state = r(n + 2, H, dim, vdim)
    w = None if mode == "fixed" else (1 + 0.1 * r(vdim if mode == "hgrn2" else hv)).to(dtype)
    gated = mode != "hgrn2"
    lower = torch.sigmoid(r(hd)).to(dtype) if mode == "hgrn2" else (1 - 2.0 ** -(3 + torch.arange(H, device=DEV) % 5).float())
    fbias, w2, b2, z = r(hd).to(dtype), (0.3 * r(hd, rank)).to(dtype), r(hd).to(dtype), r(T, hd)
    S, ref, off = state.double(), torch.empty(T, H, vdim, dtype=torch.float64, device=DEV), torch.empty(T, H, vdim, dtype=torch.float64, device=DEV)
    d = proj.double()
    for i in range(n):
        st = S[slot[i].long()].clone() if int(first[i]) else torch.zeros_like(S[0])
        for t in range(int(start[i]), int(start[i + 1])):
            q, k, v = d[t, qo:qo + hd].view(H, dim), d[t, ko:ko + hd].view(H, dim), d[t, vo:vo + hv].view(H, vdim)
            if mode == "hgrn2":
                lo = lower.double().view(H, dim)
                a = lo + (1 - lo) * torch.sigmoid(k + fbias.double().view(H, dim))
                q, k = torch.nn.functional.silu(q), 1 - a
            elif mode.startswith("gla"):
                zz = z[t].double() if mode == "gla-z" else w2.double() @ proj[t, ao:ao + rank].to(dtype).double() + b2.double()
                q, a = q * dim ** -0.5, torch.exp(torch.nn.functional.logsigmoid(zz) / 16.0).view(H, dim)
            else:
                a = lower.double().view(H, 1).expand(H, dim)
                if mode == "fixed-silu":
                    q, k, v = (torch.nn.functional.silu(x) for x in (q, k, v))
            st = st * a[:, :, None] + k[:, :, None] * v[:, None]
            o = (st * q[:, :, None]).sum(1)
            by = 1 / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5)
            if w is not None:
                by = by * (w.double().view(H, vdim) if w.numel() == hv else w.double())
            if gated:
                by = by * torch.nn.functional.silu(d[t, go:go + hv].view(H, vdim))
            ref[t], off[t] = o * by, 2.0 ** -17 * (st * q[:, :, None]).abs().sum(1).amax(-1, keepdim=True) * by.abs()
        S[slot[i].long()] = st
    modes = {"hgrn2": hops.SCAN_HGRN2, "gla": hops.SCAN_GLA, "gla-z": hops.SCAN_GLA, "fixed": hops.SCAN_FIXED, "fixed-silu": hops.SCAN_FIXED_SILU}
    out = hops.recur_step(modes[mode], proj, qo, ko, vo, go if gated else None, (ao, w2, b2) if mode == "gla" else None, z if mode == "gla-z" else None, lower, fbias, 16.0,
                          dim ** -0.5, H, dim, vdim, start, slot, first, state, w, 1e-5, dtype)
    assert float((state.double() - S).abs().max()) <= 2.0 ** -18 * float(S.abs().max())
    assert bool(((out.double().view(T, H, vdim) - ref).abs() <= off + (2.0 ** -20 if dtype == torch.float32 else 2.0 ** -8) * ref.abs()).all())


# heads on both sides of the recurrence step's limits: 36 and 37 key rows a thread, value columns that are no multiple of 4
@pytest.mark.parametrize("kind", ["gla", "hgrn2"])
@pytest.mark.parametrize("dim,vdim,fits", [(180, 176, True), (184, 176, False), (144, 208, True), (152, 208, False), (64, 130, False), (128, 256, True)])
def test_a_decode_step_serves_every_head(kind, dim, vdim, fits):
    """What the recurrence step refuses walks as before it was there.  Against 64 bits from the same bf16 weights, the low-rank decay's middle rounded to bf16 as there: the outputs are
    rounded to bf16 twice (2^-8 each of the largest), the states differ by what the middle's rounding may flip (2^-8 of a pre-activation of about 1 over tau, of a state of about 1)."""
    assert hops.recur_step_supported(dim, vdim) is fits
    H, W, T, tau = 2, 64, 3, 16.0
    g = torch.Generator(device=DEV).manual_seed(dim)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    weight = lambda n, k=W: (r(n, k) * k ** -0.5).bfloat16()
    hd, hv = H * dim, H * vdim
    w = {"q": weight(hd), "v": weight(hv), "o": torch.eye(hv, device=DEV).bfloat16(), "norm": (1 + 0.1 * r(hv if kind == "gla" else vdim)).bfloat16()}
    if kind == "gla":
        w.update({"k": weight(hd), "g": weight(hv), "a1": weight(16), "a2": weight(hd, 16), "a2.b": r(hd).bfloat16()})
    else:
        w.update({"f": weight(hd), "lower": torch.sigmoid(r(hd)).bfloat16(), "f.b": r(hd).bfloat16()})
    mixer = mixers.GatedLinearRecurrence(mixers.RecurrenceSpec(kind=kind, heads=H, dim=dim, vdim=vdim, tau=tau), w, 1e-5)
    index = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
    batch = types.SimpleNamespace(row_start=index(0, 1, 2, 3), slot=index(2, 0, 1), first_pos=index(4, 0, 9), plans={}, max_rows=1)
    state, h = r(3, H, dim, vdim), r(T, W).bfloat16()
    lin = lambda n, c: (h.double() @ w[n].double().t()).view(T, H, c)
    q, v = lin("q", dim), lin("v", vdim)
    if kind == "gla":
        k, z = lin("k", dim), (h.double() @ w["a1"].double().t()).bfloat16().double() @ w["a2"].double().t() + w["a2.b"].double()
        q, a = q * dim ** -0.5, torch.exp(torch.nn.functional.logsigmoid(z) / tau).view(T, H, dim)
    else:
        low = w["lower"].double().view(H, dim)
        a = low + (1 - low) * torch.sigmoid(lin("f", dim) + w["f.b"].double().view(H, dim))
        q, k = torch.nn.functional.silu(q), 1 - a
    S = state.double()[batch.slot.long()] * (batch.first_pos > 0).double()[:, None, None, None] * a[..., None] + k[..., None] * v[:, :, None]
    o = (S * q[..., None]).sum(2)
    o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * w["norm"].double().view(-1, vdim)
    if kind == "gla":
        o = o * torch.nn.functional.silu(lin("g", vdim))
    got = mixer.forward(h, batch, state).double().view(T, H, vdim)
    assert float((got - o).abs().max()) <= 2.0 ** -7 * float(o.abs().max())
    assert float((state.double()[batch.slot.long()] - S).abs().max()) <= 2.0 ** -8 / tau * float(S.abs().max())
