"""The sampler where its arithmetic or its grid is at an edge: a top-p that falls on the rounding of the bins' 64-bit sums, more rows than the 65535 of many grids' second dimension."""
from fractions import Fraction

import pytest
import torch

from oracle import oracle
from rtp_llm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("V", [64, 5001])
def test_top_p_within_a_rounding_of_a_bin_border(V):
    """The mass above some value is 0.75 but for half a unit of its 64-bit sum (u = 2^-53).  Added bin by bin the sum passes 0.75 with the value b of one bin, added over the
    lanes it has not passed it where the next thread's bins begin, whose values c then seem to pass it too.  Exactly: the mass before b is 0.75 - 0.43 u, b stays;
    before the first c it is 0.75 + 0.11 u, none of them stays."""
    u = 2.0 ** -53
    values = [0.75 - 2.0 ** -24, 2.0 ** -24 - 2.0 ** -48, 2.0 ** -48 - u, 0.57 * u, 0.54 * u, 0.4425 * u, 0.4400 * u]
    probs = torch.zeros(3, V)
    at = torch.randperm(V, generator=torch.Generator().manual_seed(V))[:len(values)]
    probs[:, at] = torch.tensor(values, dtype=torch.float64).float()
    mass, want = Fraction(0), torch.zeros(V, dtype=torch.bool)
    for i in at[torch.argsort(probs[0, at], descending=True)].tolist():
        want[i] = mass <= Fraction(3, 4)
        mass += Fraction(float(probs[0, i]))
    assert int(want.sum()) == 5
    ids, out = ops.top_k_top_p_sample(probs.to(DEV), torch.zeros(3, dtype=torch.int32), torch.full((3,), 0.75), torch.tensor([0.1, 0.5, 0.9]).to(DEV), return_probs=True)
    assert torch.equal(out.cpu() > 0, want.expand(3, V)) and bool(want[ids.cpu().long()].all())


@pytest.mark.parametrize("V", [3, 8])
def test_more_than_65536_rows(V):
    """65536 + 5 rows: temperature alone, temperature and penalties, and the joint form, against each row's own arithmetic (2^-22 of a value: a division and a product)."""
    B = (1 << 16) + 5
    g = torch.Generator(device=DEV).manual_seed(V)
    x, t = torch.randn(B, V, device=DEV, generator=g) * 3, torch.rand(B, device=DEV, generator=g) + 0.5
    want = x * (1.0 / (t + 1e-6))[:, None]
    got = ops.apply_penalties(x.clone(), temperature=t)
    assert bool(((got - want).abs() <= 2.0 ** -22 * want.abs()).all())
    ids = torch.randint(0, V, (B, 2), device=DEV, generator=g, dtype=torch.int32)
    pen = dict(repetition_penalty=torch.full((B,), 1.5, device=DEV), presence_penalty=torch.full((B,), 0.25, device=DEV), frequency_penalty=torch.full((B,), 0.5, device=DEV))
    count = torch.zeros_like(x).scatter_add_(1, ids.long(), torch.ones(B, 2, device=DEV))
    full = torch.where(count > 0, torch.where(want < 0, want * 1.5, want / 1.5) - 0.25 - 0.5 * count, want)
    lens = torch.full((B,), 2, dtype=torch.int32, device=DEV)
    got = ops.apply_penalties(x.clone(), temperature=t, output_ids=ids.t().contiguous(), input_lengths=lens, max_input_length=2, step=2, **pen)
    assert bool(((got - full).abs() <= 2.0 ** -21 * (full.abs() + 2)).all())
    got = ops.sampling_probs(x.clone(), t, token_ids=ids, input_lengths=lens, max_input_length=2, step=2, **pen)
    assert bool(((got - full.double().softmax(-1)).abs() <= 2.0 ** -18).all())


@pytest.mark.parametrize("step", [1, 31, 33, 700, 2048])
@pytest.mark.parametrize("kind", ["one hash", "last hash", "few ids", "one id", "outside"])
def test_history_counts(kind, step):
    """Histories whose ids share a slot of the on-chip table (probing, also over its end), repeat, or lie outside the vocabulary; every id once, by its count, in both launches that count."""
    V, B = 40000, 3
    bits = max(6, (2 * step - 1).bit_length())
    g = torch.Generator().manual_seed(step)
    ids = torch.arange(V, dtype=torch.int64)
    slot = (ids * 2654435761 % 2 ** 32) >> (32 - bits)
    pool = {"one hash": ids[slot == slot[77]], "last hash": ids[slot >= (1 << bits) - 2], "few ids": ids[5:12], "one id": ids[9:10], "outside": torch.tensor([-1, -7, 3, V, V + 9, 2 ** 31 - 1])}[kind]
    hist = pool[torch.randint(0, pool.numel(), (step, B), generator=g)].int()
    x = torch.randn(B, V, generator=g) * 3
    pen = dict(repetition_penalty=torch.tensor([1.0, 1.3, 0.7]), presence_penalty=torch.tensor([0.5, 0.0, 0.25]), frequency_penalty=torch.tensor([0.125, 0.5, 0.0]))
    lens = torch.full((B,), step, dtype=torch.int32)
    want = oracle.apply_penalties(x, output_ids=hist, input_lengths=lens, max_input_length=step, step=step, **pen)
    got = ops.apply_penalties(x.clone().to(DEV), output_ids=hist.to(DEV), input_lengths=lens, max_input_length=step, step=step, **pen)
    assert torch.equal(got.cpu(), want)
    dev = {k: v.to(DEV) for k, v in pen.items()}
    got = ops.sampling_probs(x.clone().to(DEV), token_ids=hist.t().contiguous().to(DEV), input_lengths=lens.to(DEV), max_input_length=step, step=step, **dev)
    soft = want.double().softmax(-1)            # exp2 of an argument rounded to 24 bits, |x - max| < 40 where the result counts: 40 * 2^-24 = 2.4e-6, and the sum
    assert bool(((got.cpu() - soft).abs() <= 5e-6 * soft + 1e-12).all())


@pytest.mark.parametrize("V", [700, 5001, 70001, 152064])
@pytest.mark.parametrize("kind", ["flat", "crowded k", "crowded p", "one value", "two values"])
def test_rows_with_more_values_in_a_bin_than_the_sets_hold(V, kind):
    """Multiples of 2^-34 inside one or two bins, and runs of one value: the first histogram, the second one of a bin, and the last bits over the row.  Kept sets against exact integers (the masses are
    sums of integers below 2^53)."""
    g = torch.Generator().manual_seed(V)
    n = min(V, 60000)
    if kind in ("flat", "crowded k", "crowded p"):
        # 2^18 units of 2^-34 = 2^-16 and up to 2^14 units more: a sixteenth of an octave is one bin
        units = (torch.randperm(16384, generator=g).repeat(4)[:n] if n > 16384 else torch.randperm(16384, generator=g)[:n]).long() + 262144
        if kind == "crowded k":
            units[: n // 2] = units[: n // 2] * 32 + 7
        elif kind == "crowded p":
            units[: n // 50] = units[: n // 50] * 32 + 3
    else:
        units = torch.full((n,), 262144 + 777, dtype=torch.long)
        if kind == "two values":
            units[::3] = 262144 + 778
    at = torch.randperm(V, generator=g)[:n]
    R = 4
    value = torch.zeros(V, dtype=torch.long)
    value[at] = units
    probs = (value.double() * 2.0 ** -34).float()[None].repeat(R, 1)
    assert torch.equal((probs[0].double() * 2.0 ** 34).long(), value)
    order = torch.argsort(value, descending=True, stable=True)
    before = value[order].cumsum(0) - value[order]                       # mass in front of each entry, in units
    top_k = torch.tensor([0, n // 3, n - 1, 5], dtype=torch.int32)
    want = torch.zeros(R, V, dtype=torch.bool)
    top_p = torch.empty(R)
    for r, share in enumerate((0.4, 1.0, 0.9, 0.97)):
        top_p[r] = 1.0 if share == 1.0 else float(torch.tensor(float(before[int(share * n)]) * 2.0 ** -34).float())
        keep = torch.ones(V, dtype=torch.bool)
        if 0 < int(top_k[r]) < V:
            keep &= value >= value[order[int(top_k[r]) - 1]]
        if share != 1.0:
            limit = int(round(float(top_p[r].double()) * 2 ** 34))
            inside = torch.zeros(V, dtype=torch.bool)
            inside[order[before <= limit]] = True
            keep &= inside
        want[r] = keep & (value > 0) if bool((value[keep] > 0).any()) else keep
    ids, out = ops.top_k_top_p_sample(probs.to(DEV), top_k, top_p, torch.tensor([0.0, 0.3, 0.6, 0.95]).to(DEV), return_probs=True)
    got = out.cpu() > 0
    # where equals of the border value go, the index from which they do is found from fp32 sums: their rounding (20 steps of 2^-24 of a mass of 1 to 16) is below an entry (2^-16 and up, 2^-11 there)
    assert int((got != want).sum(-1).max()) <= 1
    assert bool(got[torch.arange(R), ids.cpu().long()].all())
