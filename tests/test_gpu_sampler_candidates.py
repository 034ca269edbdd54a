"""The sampler's candidate search at its edges: how many values lie above the gathered threshold, rows that have to be searched whole, rows without alignment,
histories on both sides of the on-chip count, and the softmax that overwrites its input."""
import pytest
import torch

from oracle import oracle
from rtp_llm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("many", [1, 64, 1023, 1024, 1025, 4095, 4096, 4097, 9000])
@pytest.mark.parametrize("V", [9003, 152064])
def test_candidate_counts(many, V):
    """`many` distinct multiples of 2^-26 of one octave, spread over the row, above a floor of zeros: every partial sum is exact, so kept sets, renormalised
    values and draws equal the oracle's whatever the order of the sums."""
    g = torch.Generator().manual_seed(many * 7 + V)
    R = 5
    probs = torch.zeros(R, V)
    for r in range(R):
        at = torch.randperm(V, generator=g)[:many]
        probs[r, at] = (torch.randperm(16384, generator=g)[:many] + 16384).float() * 2.0 ** -26
    total = probs.double().sum(-1)
    top_k = torch.tensor([0, 1, many // 2 + 1, many, V + 5], dtype=torch.int32)
    top_p = torch.tensor([float(total[0]) * 0.5, 1.0, float(total[2]) * 0.9, float(total[3]) * 0.1, float(total[4]) * 2], dtype=torch.float32)
    u = torch.tensor([0.0, 0.25, 0.5, 0.75, 1023 / 1024])
    ids, out = ops.top_k_top_p_sample(probs.to(DEV), top_k, top_p, u.to(DEV), return_probs=True)
    want = oracle.top_k_top_p_filter(probs, top_k, top_p)
    assert torch.equal(out.cpu() > 0, want > 0)
    # 9000 terms of 15 bits: sums stay below 2^28 units of 2^-26, beyond fp32's 24 bits for the largest counts
    assert torch.allclose(out.cpu(), want, rtol=1e-6, atol=0)
    kept = torch.where(want > 0, probs, torch.zeros(())).double()
    c = kept.cumsum(-1) / kept.sum(-1, keepdim=True)
    for r in range(R):
        j = int(ids[r])
        assert kept[r, j] > 0 and float(c[r, j] - kept[r, j] / kept[r].sum()) - 1e-6 <= float(u[r]) <= float(c[r, j]) + 1e-6


def test_rows_that_are_searched_whole():
    """Flat rows (nothing stands out), a row of one value everywhere, an all-zero row, and a row whose largest value carries almost nothing."""
    V = 20001
    rows = [torch.full((V,), 2.0 ** -15), torch.full((V,), 2.0 ** -15), torch.zeros(V), torch.full((V,), 2.0 ** -15)]
    rows[1][:] = 2.0 ** -16 * (torch.arange(V) % 2 + 1).float()
    rows[3][7] = 2.0 ** -10
    probs = torch.stack(rows)
    top_k, top_p = torch.tensor([0, 5, 3, 0], dtype=torch.int32), torch.tensor([0.25, 1.0, 1.0, 0.5])
    u = torch.tensor([0.5, 0.5, 0.5, 0.5])
    ids, out = ops.top_k_top_p_sample(probs.to(DEV), top_k, top_p, u.to(DEV), return_probs=True)
    want = oracle.top_k_top_p_filter(probs, top_k, top_p)
    assert torch.equal(out.cpu(), want)
    assert int(ids[0]) == int(oracle.sample_rows(torch.where(want > 0, probs, torch.zeros(()))[:1], u[:1])[0]) and int(ids[2]) == V - 1


@pytest.mark.parametrize("step", [1, 3, 2047, 2048, 2049])
def test_penalties_on_both_sides_of_the_on_chip_count(step):
    g = torch.Generator().manual_seed(step)
    B, V = 3, 503
    x = torch.randn(B, V, generator=g) * 3
    ids = torch.randint(-2, V + 2, (step, B), generator=g, dtype=torch.int32)
    ids[: (step + 1) // 2, 0] = 11
    lens = torch.full((B,), max(1, step // 3), dtype=torch.int32)
    rep, pres, freq = torch.rand(B, generator=g) + 0.8, torch.rand(B, generator=g), torch.rand(B, generator=g) * 0.1
    args = dict(repetition_penalty=rep, presence_penalty=pres, frequency_penalty=freq, input_lengths=lens, max_input_length=step // 2, step=step)
    got = ops.apply_penalties(x.clone().to(DEV), output_ids=ids.to(DEV), **args).cpu()
    assert torch.equal(got, oracle.apply_penalties(x, output_ids=ids, **args))


@pytest.mark.parametrize("V", [5, 1030, 152064])
def test_softmax_over_its_own_input(V):
    x = torch.randn(3, V, generator=torch.Generator().manual_seed(V)) * 4
    want = torch.softmax(x.double(), -1)
    buf = x.to(DEV)
    out = ops.softmax_rows(buf, out=buf)
    assert out.data_ptr() == buf.data_ptr() and torch.equal(out, ops.softmax_rows(x.to(DEV)))
    assert torch.allclose(out.cpu().double(), want, rtol=5e-6, atol=1e-12)      # exp2 of an argument rounded to 24 bits: |x - max| < 40 -> 40 * 2^-24 = 2.4e-6
