"""Attention for prompt portions (matrix-core tiles) against 64-bit attention over the same bf16 pages: every instance and the guarded ones, 1 to 8 query heads per key/value
head (tiles of several sequences then share a block), portions that start inside a context, pages down to one token (more block-table entries than the kernel holds at
once), window with kept first tokens, block mask, cap, sink, gates, turned values in both layouts, a latent cache, operands off 16 bytes.
Bound: the result's rounding to bf16 (2^-9 of it, 2^-8 allowed), and queries and weights held to 2^-17 in the products: scores of |s| <= 16 move by 2^-13, a weighted
mean of values by as much of the largest value; 2^-12 allowed."""
import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops
from rtp_llm_amd.mixers import rotary_steps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [  # dim, vdim, heads, kv_heads, page, options
    (128, 128, 8, 2, 64, {}), (128, 128, 6, 3, 16, {"chunk": 100}), (128, 128, 3, 3, 64, {"window": 50}), (128, 128, 4, 1, 64, {"window": 40, "keep": 5, "gate": 1}),
    (64, 64, 4, 4, 16, {"softcap": 20.0}), (64, 64, 8, 1, 1, {}), (64, 64, 14, 2, 24, {"off": 1}), (256, 192, 8, 1, 64, {"latent": True, "sink": True}),
    (256, 192, 2, 2, 64, {}), (256, 128, 8, 1, 64, {"latent": True}), (32, 16, 3, 1, 3, {"sink": True}), (96, 112, 4, 1, 64, {"gate": 2}), (160, 208, 2, 1, 48, {"turn": 0}),
    (256, 256, 4, 1, 16, {"turn": 1, "sink": True}), (128, 128, 4, 2, 64, {"turn": 1, "gate": 2}), (64, 64, 2, 2, 64, {"turn": 0, "chunk": 64}), (32, 256, 5, 5, 1, {"off": 1, "turn": 1}),
]


@pytest.mark.parametrize("dim,vdim,H,G,page,opt", CASES)
# the last: walks that two groups of waves share and such that one keeps, also in one block
@pytest.mark.parametrize("starts,counts", [([0], [7]), ([0, 70, 250], [45, 130, 17]), ([3, 0, 0, 1, 0], [1, 2, 31, 16, 33]), ([1300], [40]), ([1300, 3, 700, 0, 590], [20, 9, 5, 16, 40])])
def test_portions(dim, vdim, H, G, page, opt, starts, counts):
    g = torch.Generator(device=DEV).manual_seed(dim + vdim + H + len(starts))
    off, n = opt.get("off", 0), len(starts)
    width = -(-(max(a + c for a, c in zip(starts, counts))) // page)
    table = torch.randperm(n * width + 2, generator=torch.Generator().manual_seed(1), dtype=torch.int32)[:n * width].reshape(n, width)
    pages = n * width + 2
    pos, seq, t0, tn, T = [], [], [], [], 0
    for s, (a, c) in enumerate(zip(starts, counts)):
        pos += list(range(a, a + c)); seq += [s] * c
        t0 += list(range(T, T + c, 16)); tn += [min(16, c - r) for r in range(0, c, 16)]
        T += c
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    cache = lambda d: torch.randn(pages * G * page * d + off, device=DEV, generator=g).bfloat16()[off:].view(pages, G, page, d)
    kc = cache(dim)
    vc = kc if opt.get("latent") else cache(vdim)
    q = torch.randn(T, H * dim + off + 3 * (off > 0), device=DEV, generator=g)[:, off:off + H * dim]
    turn, window, keep, chunk, cap = opt.get("turn"), opt.get("window", 0), opt.get("keep", 0), opt.get("chunk", 0), opt.get("softcap", 0.0)
    geom = hops.attn_geometry(H, G, dim, vdim, 0, 0, turn or 0, page, width, pages, **({"v_ld": dim} if opt.get("latent") else {}))
    vf = rotary_steps(vdim // 2, vdim, 1e4, DEV) if turn is not None else None
    sink = torch.randn(H, device=DEV, generator=g) if opt.get("sink") else None
    gate = None if not opt.get("gate") else torch.randn(T, H if opt["gate"] == 1 else H * vdim, device=DEV, generator=g)
    out = hops.attn_tiles(q, dim ** -0.5, geom, chunk, sink, vf, i32(pos), i32(seq), table.to(DEV), i32(t0), i32(tn), kc, vc, H, vdim, window=window, keep=keep, softcap=cap,
                          out_gate=gate)
    r = 0
    for s, (a, c) in enumerate(zip(starts, counts)):
        L = a + c
        use = table[s].long().to(DEV)
        k = kc[use].transpose(0, 1).reshape(G, -1, dim)[:, :L].double().repeat_interleave(H // G, 0)
        v = vc[use].transpose(0, 1).reshape(G, -1, vc.shape[-1])[:, :L, :vdim].double().repeat_interleave(H // G, 0)
        qq = q[r:r + c].double().view(c, H, dim).transpose(0, 1)
        sc = (qq @ k.transpose(1, 2).contiguous()) * dim ** -0.5
        if cap:
            sc = cap * torch.tanh(sc / cap)
        p_, key = torch.arange(a, L, device=DEV)[:, None], torch.arange(L, device=DEV)[None]
        ok = key <= p_
        if chunk:
            ok &= key >= p_ // chunk * chunk
        if window:
            ok &= (key > p_ - window) | (key < keep)
        sc = sc.masked_fill(~ok, float("-inf"))
        if sink is not None:
            sc = torch.cat([sc, sink.double()[:, None, None].expand(H, c, 1)], -1)
        ref = sc.softmax(-1)[..., :L] @ v
        if vf is not None:
            ang = p_.double() * vf.double()[None]
            c0, c1 = (slice(0, None, 2), slice(1, None, 2)) if turn == 0 else (slice(0, vdim // 2), slice(vdim // 2, None))
            x, y = ref[..., c0].clone(), ref[..., c1].clone()
            ref[..., c0], ref[..., c1] = x * ang.cos() + y * ang.sin(), y * ang.cos() - x * ang.sin()
        ref = ref.transpose(0, 1)
        if gate is not None:
            ref = ref * torch.sigmoid(gate[r:r + c].double()).view(c, H, -1)
        got = out[r:r + c].double().view(c, H, vdim)
        assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * v.abs().max()).all()), float((got - ref).abs().max())
        r += c


# grids of more than 320 blocks: one group of waves walks the keys (above, two do)
@pytest.mark.parametrize("dim,vdim,H,G,page,opt", [(128, 128, 16, 4, 64, {"chunk": 512}), (256, 192, 16, 1, 48, {"latent": True, "sink": True}), (64, 64, 16, 16, 16, {"window": 100})])
def test_portions_of_large_grids(dim, vdim, H, G, page, opt):
    test_portions(dim, vdim, H, G, page, opt, [0, 5], [1300, 70])
