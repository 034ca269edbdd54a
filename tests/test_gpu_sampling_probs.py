"""Temperature, penalties and softmax in two launches against the launches of their own, over every split of a row and slices without values: the scaled and
penalised logits are the same, the sum is formed in another order (fp32 partial sums of 1024 lanes: 2^-20 of a probability)."""
import pytest
import torch

from rtp_llm_amd import _C, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B", [1, 3, 40, 300])
@pytest.mark.parametrize("V", [1, 5, 67, 1001, 4096, 32003])
@pytest.mark.parametrize("temp,pen,step", [(True, True, 37), (True, False, 0), (False, True, 2048), (False, False, 0), (True, True, 1)])
def test_equals_separate_launches(B, V, temp, pen, step):
    if B * V > 4e6 and step > 100:
        pytest.skip("one large case of each kind is enough")
    g = torch.Generator(device=DEV).manual_seed(B + V)
    x = torch.randn(B, V, device=DEV, generator=g) * 4
    if V > 1:
        x[0, V // 2 - 1] = float("-inf")
    if V > 4:
        x[B - 1, :V - 1] = float("-inf")                       # slices without a finite value
    t = torch.rand(B, device=DEV, generator=g) + 0.5 if temp else None
    vecs = {}
    if pen:
        ids = torch.randint(-1, V + 2, (B, max(step, 1)), device=DEV, generator=g, dtype=torch.int32)
        lens = torch.randint(0, step + 1, (B,), device=DEV, generator=g, dtype=torch.int32)
        vecs = dict(repetition_penalty=torch.rand(B, device=DEV, generator=g) + 0.8, presence_penalty=torch.rand(B, device=DEV, generator=g),
                    frequency_penalty=torch.rand(B, device=DEV, generator=g), input_lengths=lens, max_input_length=step // 2, step=step)
    ref = x.clone()
    ops.apply_penalties(ref, temperature=t, **(dict(vecs, output_ids=ids.t().contiguous()) if pen else {}))
    ref = ops.softmax_rows(ref)
    got = ops.sampling_probs(x.clone(), t, **(dict(vecs, token_ids=ids) if pen else {}))
    assert bool(((got - ref).abs() <= 2.0 ** -20 * ref + 1e-30).all()) and torch.equal(got == 0, ref == 0)


def test_long_histories_are_refused():
    x = torch.zeros(1, 8, device=DEV)
    one = torch.ones(1, device=DEV)
    with pytest.raises(_C.Mi355Error):
        ops.sampling_probs(x, None, one, one, one, torch.zeros(1, 2049, dtype=torch.int32, device=DEV), None, 0, 2049)


@pytest.mark.parametrize("V", [3, 67, 4096, 32003, 152064])
def test_rows_with_infinities_and_nans(V):
    """+infinity or NaN among a row's logits, wherever its slice lies, and a row without a finite value: NaN all over the row, as from the launches of their own; the other rows
    are what they are without them, and a draw stays in the vocabulary."""
    g = torch.Generator(device=DEV).manual_seed(V)
    clean = torch.randn(9, V, device=DEV, generator=g) * 4
    x, t = clean.clone(), torch.rand(9, device=DEV, generator=g) + 0.5
    x[1, 0], x[2, V - 1], x[3, V // 2] = float("inf"), float("inf"), float("nan")
    x[5, V - 1], x[5, 0], x[6], x[7] = float("nan"), float("inf"), float("-inf"), float("nan")
    ref = x.clone()
    ops.apply_penalties(ref, temperature=t)
    ref = ops.softmax_rows(ref)
    got, want = ops.sampling_probs(x.clone(), t), ops.sampling_probs(clean.clone(), t)
    bad = torch.tensor([r in (1, 2, 3, 5, 6, 7) for r in range(9)], device=DEV)
    assert bool(ref[bad].isnan().all()) and bool(got[bad].isnan().all()) and torch.equal(got[~bad], want[~bad])
    ids = [ops.top_k_top_p_sample(p.clone(), torch.full((9,), 5, dtype=torch.int32), torch.full((9,), 0.9), torch.full((9,), 0.4, device=DEV)) for p in (got, want)]
    assert torch.equal(ids[0][~bad], ids[1][~bad]) and bool(((ids[0] >= 0) & (ids[0] < V)).all())
