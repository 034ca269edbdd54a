"""hy_walk's tiles of 16 tokens in the forms that scan may pick, forced here: whole and in chunks, every mode, around the tile's and the chunk's edges, keys and values that fill no
16 or 64.  Errors as in test_gpu_walk.py: the 2-norm over that of the same walk of absolute values, 3 sqrt(32) 2^-24 = 1e-6; a constant decay of at most 0.96 remembers 32 tokens too.
An infinite or undefined value reaches its own token's outputs and later ones, no earlier ones and no other head or column."""
import pytest
import torch

from rtp_llm_amd import _C, hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(monkeypatch, C, mode, proj, qo, ko, vo, z, lower, fbias, tau, H, dim, vdim, starts, slot, first, state, longest):
    monkeypatch.setattr(hops, "gated_form", lambda *a: C)
    monkeypatch.setattr(hops, "tiles_form", lambda *a: C)
    monkeypatch.setattr(hops, "FIXED_TILES_FROM", 0)
    return hops.scan(mode, proj, qo, ko, vo, z, lower, fbias, tau, dim ** -0.5, H, dim, vdim, starts, slot, first, state, torch.bfloat16, plans={}, max_rows=longest)


@pytest.mark.parametrize("mode,tau", [(hops.SCAN_GLA, 16.0), (hops.SCAN_GLA, 1.0), (hops.SCAN_HGRN2, 1.0), (hops.SCAN_FIXED, 1.0), (hops.SCAN_FIXED_SILU, 1.0)])
@pytest.mark.parametrize("H,dim,vdim,off", [(2, 64, 128, 0), (1, 5, 3, 1), (3, 17, 48, 2), (2, 65, 33, 1), (1, 128, 144, 0)])
@pytest.mark.parametrize("C", [0, 32])
def test_forms(monkeypatch, mode, tau, H, dim, vdim, off, C):
    lens = [1, 15, 16, 17, 33, 65, 97]
    g = torch.Generator(device=DEV).manual_seed(dim + vdim)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T, n = sum(lens), len(lens)
    proj, z = r(T, off + 2 * H * dim + H * vdim + 3), r(T, H * dim) + 2
    fixed = mode in (hops.SCAN_FIXED, hops.SCAN_FIXED_SILU)
    lower = torch.linspace(0.5, 0.96, H, device=DEV) if fixed else torch.rand(H * dim, device=DEV, generator=g).bfloat16()
    fbias = r(H * dim).bfloat16()
    qo, ko, vo = off, off + H * dim, off + 2 * H * dim
    slot = torch.randperm(n + 1, device=DEV, generator=g)[:n].int()
    first = torch.tensor([0 if i % 2 else 9 for i in range(n)], dtype=torch.int32, device=DEV)
    starts = torch.tensor([sum(lens[:i]) for i in range(n + 1)], dtype=torch.int32, device=DEV)
    state = r(n + 1, H, dim, vdim)
    before = state.clone()
    out = _run(monkeypatch, C, mode, proj, qo, ko, vo, z, lower, fbias, tau, H, dim, vdim, starts, slot, first, state, max(lens))
    d = lambda o, c: proj[:, o:o + H * c].double().view(T, H, c)
    silu = torch.nn.functional.silu
    q, k, v = d(qo, dim), d(ko, dim), d(vo, vdim)
    if mode == hops.SCAN_GLA:
        q, a = q * dim ** -0.5, torch.exp(torch.nn.functional.logsigmoid(z.double()) / tau).view(T, H, dim)
    elif mode == hops.SCAN_HGRN2:
        low = lower.double().view(H, dim)
        a = low + (1 - low) * torch.sigmoid(k + fbias.double().view(H, dim))
        q, k = silu(q), 1 - a
    else:
        a = lower.double()[None, :, None].expand(T, H, dim)
        if mode == hops.SCAN_FIXED_SILU:
            q, k, v = silu(q), silu(k), silu(v)

    def walk(q, k, v, S):
        o = []
        for t in range(lo, hi):
            S = S * a[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
            o.append((S * q[t][:, :, None]).sum(1))
        return torch.stack(o), S

    rel = lambda x, y, scale: float((x.double() - y).norm() / scale.norm())
    for i in range(n):
        lo, hi = int(starts[i]), int(starts[i + 1])
        S0 = before[int(slot[i])].double() * (int(first[i]) > 0)
        o, S = walk(q, k, v, S0)
        o_abs, S_abs = walk(q.abs(), k.abs() + (mode == hops.SCAN_HGRN2), v.abs(), S0.abs())
        assert rel(out[lo:hi].view(hi - lo, H, vdim), o, o_abs) < 1e-6
        assert rel(state[int(slot[i])], S, S_abs) < 1e-6
    unused = [i for i in range(n + 1) if i not in slot.tolist()]
    assert torch.equal(state[unused], before[unused])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("C", [0, 32])
def test_undefined_values_stay_behind_their_token(monkeypatch, C, bad):
    H, dim, vdim, T, at = 2, 64, 64, 70, 41
    g = torch.Generator(device=DEV).manual_seed(1)
    proj, z = torch.randn(T, 2 * H * dim + H * vdim, device=DEV, generator=g), torch.randn(T, H * dim, device=DEV, generator=g) + 2
    index = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
    outs = []
    for x in (None, bad):
        p = proj.clone()
        if x is not None:
            p[at, 2 * H * dim + 5] = x                     # head 0, column 5
        outs.append(_run(monkeypatch, C, hops.SCAN_GLA, p, 0, H * dim, 2 * H * dim, z, None, None, 16.0, H, dim, vdim, index(0, T), index(0), index(0),
                         torch.zeros(1, H, dim, vdim, device=DEV), T))
    good, odd = outs
    assert torch.equal(good[:at], odd[:at]) and not torch.isfinite(odd[at:, 5]).any()
    rest = [c for c in range(H * vdim) if c != 5]
    tol = 1e-6 * float(good.abs().max()) * dim ** 0.5      # the tile with the bad value sums its products in another order
    assert float((good[:, rest] - odd[:, rest]).abs().max()) < tol


@pytest.mark.parametrize("tau", [4.0, 16.0, 64.0])
@pytest.mark.parametrize("lo,hi", [(-90.0, -30.0), (-30.0, -2.0), (-2.0, 8.0)])
def test_decay_of_a_token(tau, lo, hi):
    """sigmoid(z)^(1 / tau), tau a power of two so that the division is exact.  Bound in units of 2^-24: the exponential's last place 2, log(1 + e^-|z|) below 0.7 to two of its places
    3 / tau, and where it is not lost beside z (above -18) the rounding of their sum |z| / tau."""
    H, dim, n = 2, 64, 500
    z = torch.rand(n, H * dim, device=DEV, dtype=torch.float64, generator=torch.Generator(device=DEV).manual_seed(int(tau))).mul(hi - lo).add(lo).float()
    proj, state, decay = torch.ones(n, 2 * H * dim + H * 8, device=DEV), torch.zeros(n, H, dim, 8, device=DEV), torch.zeros(n, H, dim, device=DEV)
    at = torch.arange(n + 1, dtype=torch.int32, device=DEV)              # a sequence each: the product of its decays is that of its token
    first = torch.zeros(n, dtype=torch.int32, device=DEV)
    _C.check_hybrid(_C.hybrid_lib().mi355_hy_walk(hops.SCAN_GLA, proj.data_ptr(), proj.stride(0), 0, H * dim, 2 * H * dim, z.data_ptr(), H * dim, None, None, tau, 1.0, H, dim, 8,
                                                  at.data_ptr(), at.data_ptr(), first.data_ptr(), n, state.data_ptr(), None, decay.data_ptr(), 0, hops.act_code(torch.bfloat16),
                                                  torch.cuda.current_stream().cuda_stream), "hy_walk")
    ref = torch.exp(torch.nn.functional.logsigmoid(z.double()) / tau)
    bound = 2.0 ** -24 * (2 + 3 / tau + torch.where(z > -18, z.abs(), 0.0).double() / tau)
    off = (decay.view(n, H * dim).double() / ref - 1).abs()
    assert bool((off <= bound)[ref > 1e-30].all())


def test_decay_at_the_ends():
    n, dim = 6, 4
    z = torch.tensor([float("inf"), float("-inf"), -1e30, 1e30, 0.0, float("nan")], device=DEV)[:, None].expand(n, dim).contiguous()
    proj, state, decay = torch.ones(n, 12, device=DEV), torch.zeros(n, 1, dim, 4, device=DEV), torch.zeros(n, dim, device=DEV)
    at, first = torch.arange(n + 1, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
    for tau in (1.0, 16.0):
        _C.check_hybrid(_C.hybrid_lib().mi355_hy_walk(hops.SCAN_GLA, proj.data_ptr(), 12, 0, 4, 8, z.data_ptr(), dim, None, None, tau, 1.0, 1, dim, 4, at.data_ptr(), at.data_ptr(),
                                                      first.data_ptr(), n, state.data_ptr(), None, decay.data_ptr(), 0, hops.act_code(torch.bfloat16),
                                                      torch.cuda.current_stream().cuda_stream), "hy_walk")
        got = decay[:, 0].tolist()
        assert got[:4] == [1.0, 0.0, 0.0, 1.0] and abs(got[4] - 0.5 ** (1 / tau)) < 1e-6 and got[5] != got[5]


@pytest.mark.parametrize("mode,tau,mean,width", [(hops.SCAN_GLA, 1.0, 0.0, 2.0), (hops.SCAN_GLA, 1.0, 2.0, 2.0), (hops.SCAN_GLA, 16.0, -10.0, 6.0), (hops.SCAN_GLA, 16.0, 3.0, 2.0),
                                                 (hops.SCAN_HGRN2, 1.0, 0.0, 1.0), (hops.SCAN_FIXED, 1.0, 0.0, 1.0)])
@pytest.mark.parametrize("dim,C", [(64, 0), (64, 32), (128, 64)])
def test_no_further_off_than_token_by_token(monkeypatch, mode, tau, mean, width, dim, C):
    """Decays that forget within a tile and such that remember for hundreds of tokens.  Token by token a state takes a rounding of every product and one of every sum; a tile's products
    round their key once and add in order, so its error is no larger: 10 % of room for what 3 runs of random roundings differ by (measured 0.60 to 1.06; with a tile's tokens added
    out of order 1.24).  Outputs sum 64 or 128 products either way, 5 % (measured 0.66 to 0.97)."""
    H, vdim, T = 8, 128, 700
    errors = torch.zeros(2, 2, dtype=torch.float64)                      # [tiles, token by token][outputs, states]
    for seed in range(3):
        g = torch.Generator(device=DEV).manual_seed(seed)
        r = lambda *s: torch.randn(*s, device=DEV, generator=g)
        proj, z = r(T, 2 * H * dim + H * vdim), r(T, H * dim) * width + mean
        fixed = mode == hops.SCAN_FIXED
        lower = torch.linspace(0.6, 0.99, H, device=DEV) if fixed else (torch.rand(H * dim, device=DEV, generator=g) * 0.5 + 0.5).bfloat16()
        fbias = r(H * dim).bfloat16()
        index = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
        d = lambda o, c: proj[:, o:o + H * c].double().view(T, H, c)
        q, k, v = d(0, dim), d(H * dim, dim), d(2 * H * dim, vdim)
        if mode == hops.SCAN_GLA:
            q, a = q * dim ** -0.5, torch.exp(torch.nn.functional.logsigmoid(z.double()) / tau).view(T, H, dim)
        elif mode == hops.SCAN_HGRN2:
            low = lower.double().view(H, dim)
            a = low + (1 - low) * torch.sigmoid(k + fbias.double().view(H, dim))
            q, k = torch.nn.functional.silu(q), 1 - a
        else:
            a = lower.double()[None, :, None].expand(T, H, dim)
        S, o = torch.zeros(H, dim, vdim, dtype=torch.float64, device=DEV), []
        for t in range(T):
            S = S * a[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
            o.append((S * q[t][:, :, None]).sum(1))
        o = torch.stack(o)
        for way in range(2):
            state = torch.zeros(1, H, dim, vdim, device=DEV)
            args = (mode, proj, 0, H * dim, 2 * H * dim, z, lower, fbias, tau)
            if way == 0:
                out = _run(monkeypatch, C, *args, H, dim, vdim, index(0, T), index(0), index(0), state, T)
            else:
                out = hops.scan(*args, dim ** -0.5, H, dim, vdim, index(0, T), index(0), index(0), state, torch.bfloat16, chunked=False, max_rows=T)
            errors[way] += torch.stack([((out.view(T, H, vdim).double() - o).norm() / o.norm()), (state[0].double() - S).norm() / S.norm()]).cpu()
    assert errors[0, 0] <= 1.05 * errors[1, 0] and errors[0, 1] <= 1.1 * errors[1, 1], errors.tolist()
