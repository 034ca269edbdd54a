"""Routing with a lane for each expert and the sort of up to 64 experts, against the rule written out: eligible experts by score, ties to the lower index."""
import math

import pytest
import torch

from rtp_llm_amd import hybrid_ops as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _route(z, groups, keep, top, score, group_top, scale):
    T, E = z.shape
    zd = z.double()
    m = zd.amax(-1, keepdim=True)
    s = torch.sigmoid(zd) if score == "sigmoid" else torch.exp(zd - m)
    if score == "softmax":
        s = s / s.sum(-1, keepdim=True)
    per, ids, wts = E // groups, [], []
    # what ranks: logits, of which the scores are monotone functions (fp32 scores may tie where logits do not, so softmax ranks are by fp32 scores)
    key = z if score != "softmax" else torch.softmax(z, -1)
    for t in range(T):
        g = [sorted((float(v) for v in s[t, i * per:(i + 1) * per]), reverse=True) for i in range(groups)]
        best = [sum(v[:2]) if group_top == 2 and per >= 2 else v[0] for v in g]
        kept = sorted(range(groups), key=lambda i: (-best[i], i))[:keep] if groups > 1 and keep < groups else range(groups)
        e = sorted((e for e in range(E) if e // per in kept), key=lambda e: (-float(key[t, e]), e))[:top]
        w = s[t, e] * scale
        ids.append(e)
        wts.append(w / s[t, e].sum() if score == "chosen" else w)
    return torch.tensor(ids), torch.stack(wts)


@pytest.mark.parametrize("E,groups,keep,top", [(16, 4, 2, 4), (16, 1, 1, 2), (3, 1, 1, 3), (8, 8, 3, 3), (24, 4, 2, 6), (32, 1, 1, 8), (40, 5, 2, 9), (64, 8, 4, 8), (64, 1, 1, 64), (1, 1, 1, 1),
                                                (72, 8, 4, 8)])
@pytest.mark.parametrize("score,group_top", [("softmax", 1), ("sigmoid", 2), ("chosen", 1)])
@pytest.mark.parametrize("T", [65, 333])
def test_route_and_sort(E, groups, keep, top, score, group_top, T):
    g = torch.Generator().manual_seed(E * 7 + T)
    z = torch.randn(T, E, generator=g) * 2
    z[: T // 2] = (z[: T // 2] * 2).round() / 2                                 # ties
    if score != "softmax" and E > top:
        z[3, 0] = -math.inf
    wide = torch.zeros(T, E + 5, device=DEV)
    wide[:, :E] = z.to(DEV)
    kw = dict(sigmoid=score == "sigmoid", chosen=score == "chosen", group_top=group_top, scale=1.25)
    ahead = torch.zeros(1 << 22, dtype=torch.bfloat16, device=DEV)
    ids, wts, offs, src, place, tiles = (t.cpu() for t in hops.moe_route_sorted(wide[:, :E], E, groups, keep, top, ahead=ahead, **kw))
    ref_ids, ref_wts = _route(z, groups, keep, top, score, group_top, 1.25)
    assert torch.equal(ids.long(), ref_ids)
    # relative, in units of 2^-24: the difference of two logits up to 16 apart (16), exp (4), a sum of up to 64 terms one by one (63) and of the score's own terms in a tree (6), quotients (2)
    assert bool(((wts.double() - ref_wts).abs() <= 91 * 2.0 ** -24 * ref_wts + 1e-37).all())
    _sorted(ids, E, top, offs, src, place, tiles)
    again, w2 = hops.moe_route(wide[:, :E], groups, keep, top, **kw)
    assert torch.equal(again.cpu(), ids) and torch.equal(w2.cpu(), wts)


def _sorted(ids, E, top, offs, src, place, tiles):
    n, flat = ids.numel(), ids.flatten().long()
    count = torch.bincount(flat, minlength=E)
    assert torch.equal(offs.long(), torch.cat([torch.zeros(1, dtype=torch.long), count.cumsum(0)]))
    assert torch.equal(place.sort().values.long(), torch.arange(n))
    assert torch.equal(src[place.long()].long(), torch.arange(n) // top)
    assert bool(((place >= offs[flat]) & (place < offs[flat + 1])).all())
    want = [(e, int(offs[e]) + 64 * m) for e in range(E) for m in range(-(-int(count[e]) // 64))]
    assert int(tiles[0]) == len(want) and tiles[1:1 + 2 * len(want)].view(-1, 2).tolist() == [list(t) for t in want]


@pytest.mark.parametrize("E", [1, 16, 63, 64, 65])
@pytest.mark.parametrize("T,top", [(1, 1), (1024, 1), (1025, 1), (2048, 4), (2049, 4), (8192, 4), (8193, 4)])      # one round of the block, its 8 and 32 rounds, and more
def test_sort(E, T, top):
    g = torch.Generator().manual_seed(E + T)
    ids = (torch.rand(T, top, generator=g) ** 3 * E).int().clamp_(max=E - 1)
    _sorted(ids, E, top, *(t.cpu() for t in hops.moe_align(ids.to(DEV), E)))


def test_logits_that_are_no_numbers_route_within_range():
    z = torch.randn(70, 16, device=DEV)
    z[5], z[6, 3], z[7, :15] = math.nan, math.nan, math.nan
    for kw in ({}, dict(sigmoid=True, group_top=2), dict(chosen=True)):
        ids = hops.moe_route(z, 4, 2, 4, **kw)[0].long().cpu()
        assert all(len(set(r)) == 4 and 0 <= min(r) and max(r) < 16 for r in ids.tolist())
