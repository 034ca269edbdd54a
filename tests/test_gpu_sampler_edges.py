"""The sampler where its arithmetic or its grid is at an edge: a top-p that falls on the rounding of the bins' 64-bit sums, more rows than the 65535 of many grids' second dimension."""
from fractions import Fraction

import pytest
import torch

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
