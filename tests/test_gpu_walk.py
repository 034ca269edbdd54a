"""The gated recurrences (GLA, HGRN2) over prompt portions, whole and in chunks, against a 64-bit walk: key and value sizes around the kernel's patches, unaligned
projections, ragged sequences from one token up, fresh and continued states.  Error in the 2-norm over that of the same walk of absolute values: a rounding (2^-24) per
product, per sum and per decay, a state remembering about 1 / (1 - a) <= 32 tokens in the root mean square, so 3 sqrt(32) 2^-24 = 1e-6.  HGRN2's key 1 - a has the rounding
of 1, not its own, so its scale is taken with |k| + 1."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _walk64(q, k, v, a, S):
    o = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=torch.float64, device=q.device)
    for t in range(q.shape[0]):
        S = S * a[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
        o[t] = (S * q[t][:, :, None]).sum(1)
    return o, S


@pytest.mark.parametrize("mode", [hops.SCAN_GLA, hops.SCAN_HGRN2])
@pytest.mark.parametrize("H,dim,vdim,off", [(2, 64, 128, 0), (3, 8, 4, 0), (2, 40, 72, 4), (1, 61, 30, 1), (2, 72, 136, 0), (1, 128, 200, 3), (1, 127, 129, 2)])
@pytest.mark.parametrize("lens", [[1, 1, 1], [300], [33, 700, 1, 129], [16, 17, 32, 15], [40] * 130])
def test_gated_walk(mode, H, dim, vdim, off, lens):
    g = torch.Generator(device=DEV).manual_seed(dim * vdim + len(lens))
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T, n = sum(lens), len(lens)
    width = off + 2 * H * dim + H * vdim + 5
    proj, z = r(T, width), r(T, H * dim + off)[:, off:]
    lower, fbias = torch.rand(H * dim, device=DEV, generator=g).bfloat16(), r(H * dim).bfloat16()
    qo, ko, vo = off, off + H * dim, off + 2 * H * dim
    slot = torch.randperm(n + 2, device=DEV, generator=g)[:n].int()
    first = torch.tensor([0 if i % 2 == 0 else 7 for i in range(n)], dtype=torch.int32, device=DEV)
    starts = torch.tensor([sum(lens[:i]) for i in range(n + 1)], dtype=torch.int32, device=DEV)
    state = r(n + 2, H, dim, vdim)
    before = state.clone()
    out = hops.scan(mode, proj, qo, ko, vo, z if mode == hops.SCAN_GLA else None, lower if mode == hops.SCAN_HGRN2 else None, fbias if mode == hops.SCAN_HGRN2 else None,
                    16.0, dim ** -0.5, H, dim, vdim, starts, slot, first, state, torch.bfloat16, plans={}, max_rows=max(lens))
    d = lambda o, c: proj[:, o:o + H * c].double().view(T, H, c)
    q, k, v = d(qo, dim), d(ko, dim), d(vo, vdim)
    if mode == hops.SCAN_GLA:
        q, a = q * dim ** -0.5, torch.exp(torch.nn.functional.logsigmoid(z.double()) / 16.0).view(T, H, dim)
    else:
        low = lower.double().view(H, dim)
        a = low + (1 - low) * torch.sigmoid(k + fbias.double().view(H, dim))
        q, k = torch.nn.functional.silu(q), 1 - a
    for i in range(n):
        lo, hi = int(starts[i]), int(starts[i + 1])
        S0 = before[int(slot[i])].double() if int(first[i]) else torch.zeros(H, dim, vdim, dtype=torch.float64, device=DEV)
        o, S = _walk64(q[lo:hi], k[lo:hi], v[lo:hi], a[lo:hi], S0)
        o_abs, S_abs = _walk64(q[lo:hi].abs(), k[lo:hi].abs() + (mode == hops.SCAN_HGRN2), v[lo:hi].abs(), a[lo:hi], S0.abs())
        rel = lambda x, y, scale: float((x.double() - y).norm() / scale.norm())
        assert rel(out[lo:hi].view(hi - lo, H, vdim), o, o_abs) < 1e-6
        assert rel(state[int(slot[i])], S, S_abs) < 1e-6
        if i >= 3:
            break                                        # the 64-bit walk is a Python loop
    untouched = torch.ones(n + 2, dtype=torch.bool, device=DEV)
    untouched[slot.long()] = False
    assert torch.equal(state[untouched], before[untouched])
