"""The sampler's four joint launches against its two separate ones (softmax of the penalised logits, then the filter and the draw on whole rows)."""
import pytest
import torch

from rtp_llm_amd import ops, sampler

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _logits(kind, B, V, g):
    x = torch.randn(B, V, device=DEV, generator=g) * 2.0
    if kind == "peaked":                      # a few dozen candidates above a bulk
        n = min(V, 48)
        x.scatter_(1, torch.rand(B, V, device=DEV, generator=g).topk(n).indices, 8.0 + 2.5 * torch.randn(B, n, device=DEV, generator=g))
    elif kind == "flat":                      # more values than a list holds
        x *= 0.05
    elif kind == "ties":
        x = x.round()
    elif kind == "masked":                    # -inf and the type's lowest value beside few finite ones
        x[torch.rand(B, V, device=DEV, generator=g) < 0.5] = float("-inf")
        x[torch.rand(B, V, device=DEV, generator=g) < 0.5] = torch.finfo(torch.float32).min
        x[:, V // 2] = 3.0
    elif kind == "spike":                     # one token has all the mass that a float holds
        x[:, V // 3] = 200.0
    return x


# rows of one slice and of sixteen, slices held in registers (up to 20480 values) and walked, rows off 16 bytes, a vocabulary below one load, rows of one round of
# launches and one more, of three
@pytest.mark.parametrize("B,V", [(1, 7), (3, 1000), (2, 8191), (5, 32001), (1, 152064), (64, 20484), (300, 4099), (2, 400003), (1025, 100), (2100, 33)])
@pytest.mark.parametrize("kind", ["peaked", "flat", "ties", "masked", "spike"])
def test_joint_draw_equals_separate_launches(B, V, kind):
    g = torch.Generator(device=DEV).manual_seed(B * 1000 + V)
    x = _logits(kind, B, V, g)
    pick = lambda values, dt: torch.tensor(values, dtype=dt, device=DEV)[torch.randint(0, len(values), (B,), device=DEV, generator=g)]
    k, p = pick([0, 1, 7, 50, 3000, V], torch.int32), pick([0.0, 0.3, 0.8, 0.95, 0.999999, 1.0, -0.5], torch.float32)
    u = torch.rand(B, device=DEV, generator=g) * 0.996 + 0.002
    hist = torch.randint(-1, V + 2, (B, 40), dtype=torch.int32, device=DEV, generator=g)
    pen = dict(repetition_penalty=pick([1.0, 1.2], torch.float32), presence_penalty=pick([0.0, 0.4], torch.float32), frequency_penalty=pick([0.0, 0.1], torch.float32),
               token_ids=hist, input_lengths=torch.full((B,), 40, dtype=torch.int32, device=DEV), max_input_length=40, step=40)
    for t, kw in ((None, {}), (pick([0.6, 1.0], torch.float32), pen)):
        want = ops.sampling_probs(x.clone(), t, **kw)
        want_ids = ops.top_k_top_p_sample(want, k, p, u)
        got = x.clone()
        ids = ops.sampling_draw(got, k, p, u, t, **kw)
        assert torch.equal(got.view(torch.int32), want.view(torch.int32)), "the probabilities are the same launch's"
        # a draw may land on the neighbour where the fp32 sums of whole rows and the exact ones of the list differ in the last bit; none does at these seeds
        assert torch.equal(ids, want_ids), (k[ids != want_ids], p[ids != want_ids])


def test_joint_draw_takes_kept_tokens_only():
    """Uniforms at both ends of the range: the first and the last token that the filter keeps, of a row with a known order."""
    V, B = 5000, 4
    x = torch.full((B, V), -20.0, device=DEV)
    x[:, 1234], x[:, 77], x[:, 4000], x[:, 9] = 5.0, 4.0, 3.0, 2.0
    k = torch.tensor([3, 3, 0, 0], dtype=torch.int32, device=DEV)
    p = torch.tensor([1.0, 1.0, 0.85, 0.85], device=DEV)          # 0.644, 0.237, 0.087, 0.032: the third starts above 0.85
    u = torch.tensor([0.0, 0.9999999, 0.0, 0.9999999], device=DEV)
    assert ops.sampling_draw(x, k, p, u).tolist() == [77, 4000, 77, 1234]


@pytest.mark.parametrize("top_k,top_p,joint", [(0, 1.0, False), (300, 1.0, False), (0, 0.0, False), (50, 1.0, True), (0, 0.9, True), (299, 1.0, True)])
def test_rows_without_a_filter_take_the_separate_launches(monkeypatch, top_k, top_p, joint):
    """sample_greedy: top-k of 0 or the whole row and top-p of 1 (0 means that too) keep everything; one row with a filter is enough for the joint draw."""
    B, V = 3, 300
    x = torch.randn(B, V, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)) * 2
    calls = []
    one, two = ops.sampling_draw, ops.top_k_top_p_sample
    monkeypatch.setattr(ops, "sampling_draw", lambda *a, **k: calls.append("joint") or one(*a, **k))
    monkeypatch.setattr(ops, "top_k_top_p_sample", lambda *a, **k: calls.append("separate") or two(*a, **k))
    k, p, u = torch.tensor([0, top_k, 0], dtype=torch.int32), torch.tensor([1.0, top_p, 1.0]), torch.tensor([0.2, 0.5, 0.9])
    logits = x.clone()
    ids = sampler.sample_greedy(sampler.GreedyParams(logits=logits, input_lengths=torch.ones(B, dtype=torch.int32), sequence_lengths=torch.ones(B, dtype=torch.int32),
                                                     token_ids=torch.zeros(B, 2, dtype=torch.int32), step=1, top_k=k, top_p=p, temperature=torch.ones(B), uniform=u))
    assert calls == ["joint" if joint else "separate"]
    probs = ops.sampling_probs(x.clone())
    assert torch.equal(logits, probs) and torch.equal(ids, two(probs, k.to(DEV), p.to(DEV), u.to(DEV)))


# a row is not counted from 8193 values on, where they are equal; one more value here and there, half of a row masked
@pytest.mark.parametrize("B,V", [(2, 8192), (2, 8193), (70, 8200), (3, 32001), (2, 152064)])
@pytest.mark.parametrize("kind", ["equal", "one above", "half masked", "beside others"])
def test_rows_too_flat_to_count(B, V, kind):
    x = torch.full((B, V), 1.5, device=DEV)
    if kind == "one above":
        x[:, V // 3] = 2.0
    elif kind == "half masked":
        x[:, ::2] = float("-inf")
    elif kind == "beside others":
        x[1:] = torch.randn(B - 1, V, device=DEV, generator=torch.Generator(device=DEV).manual_seed(V)) * 3
    k, u = torch.zeros(B, dtype=torch.int32, device=DEV), torch.linspace(0.01, 0.99, B, device=DEV)
    for p in (0.3141, 0.9017):                # between two prefixes of equal values: their fp32 and exact sums keep as many
        p = torch.full((B,), p, device=DEV)
        want = ops.sampling_probs(x.clone())
        got = x.clone()
        ids = ops.sampling_draw(got, k, p, u)
        assert torch.equal(got, want) and torch.equal(ids, ops.top_k_top_p_sample(want, k, p, u))


def _step_params(B, V, n, pen, plain_t, seed):
    g = torch.Generator().manual_seed(seed)
    pick = lambda values: torch.tensor(values)[torch.randint(0, len(values), (B,), generator=g)]
    p = dict(top_k=pick([0, 1, 5, V, V + 3]).int(), top_p=pick([0.0, 1e-8, -1e-8, 0.4, 0.9, 1.0]).float(), temperature=torch.ones(B) if plain_t else pick([0.5, 1.0, 1.5]).float(),
             uniform=torch.rand(B, generator=g))
    p["top_k"][0], p["top_p"][0] = 7, 0.8                         # one row at least has a filter
    if pen != "none":
        on = pen == "on"
        p.update(repetition_penalty=pick([1.0, 1.3] if on else [1.0]).float(), presence_penalty=pick([0.0, 0.4] if on else [0.0]).float(), frequency_penalty=pick([0.0, -0.2] if on else [0.0]).float())
    lens = torch.randint(0, n + 1, (B,), generator=g, dtype=torch.int32)
    return p, torch.randint(0, V, (B, n + 1), generator=g, dtype=torch.int32), lens, torch.randint(0, n + 1, (B // 2,), generator=g, dtype=torch.int32)


@pytest.mark.parametrize("B,V,n", [(1, 50, 0), (3, 1000, 1), (64, 4099, 40), (5, 300, 2047), (7, 300, 2048)])
@pytest.mark.parametrize("pen", ["none", "neutral", "on"])
@pytest.mark.parametrize("plain_t", [True, False])
def test_step_from_host_vectors(monkeypatch, B, V, n, pen, plain_t):
    """sample_greedy on host vectors, in one native call up to a history of 2047, against its general path: the same ids, probabilities and history, also where a tensor has another type or
    strides (which the native call leaves to that path)."""
    x = torch.randn(B, V, device=DEV, generator=torch.Generator(device=DEV).manual_seed(n)) * 3
    vectors, taken = ops.sampler_vectors, []

    def run(native, change=lambda p: p):
        monkeypatch.setattr(ops, "sampler_vectors", (lambda *a: taken.append(vectors(*a)) or taken[-1]) if native else (lambda *a: None))
        p, tokens, lens, seqs = _step_params(B, V, n, pen, plain_t, B + n)
        logits = x.clone()
        ids = sampler.sample_greedy(sampler.GreedyParams(logits=logits, input_lengths=lens, sequence_lengths=seqs, token_ids=tokens, step=n, **change(p)))
        return ids.tolist(), logits, tokens

    want = run(False)
    for change in (lambda p: p, lambda p: {**p, "top_p": p["top_p"].double()}, lambda p: {**p, "top_k": torch.stack([p["top_k"], p["top_k"]], 1)[:, 0]}):
        got = run(True, change)
        assert got[0] == want[0] and torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    assert [t is not None for t in taken] == [n < 2048, False, B == 1 and n < 2048]


@pytest.mark.parametrize("n,top_k,pen", [(3, 0, False), (3, 1, True), (3, 0, True), (2048, 5, True), (2100, 0, False)])
def test_steps_that_stay_general(monkeypatch, n, top_k, pen):
    """Steps without a filter never have their vectors built for the native call, and those past its history are turned away before a vector is looked at: ids, probabilities and history as without
    the question."""
    B, V = 6, 500
    x = torch.randn(B, V, device=DEV, generator=torch.Generator(device=DEV).manual_seed(n)) * 3
    built, vectors, filters = [], ops.sampler_vectors, ops.sampler_filters

    def run(native):
        monkeypatch.setattr(ops, "sampler_vectors", (lambda *a: built.append(vectors(*a))) if native else (lambda *a: None))
        monkeypatch.setattr(ops, "sampler_filters", filters if native else (lambda *a: None))
        g = torch.Generator().manual_seed(n)
        p = dict(top_k=torch.full((B,), top_k, dtype=torch.int32), top_p=torch.ones(B), temperature=torch.full((B,), 0.7), uniform=torch.rand(B, generator=g))
        if pen:
            p.update(repetition_penalty=torch.full((B,), 1.3), presence_penalty=torch.full((B,), 0.2), frequency_penalty=torch.zeros(B))
        tokens, lens = torch.randint(0, V, (B, n + 1), generator=g, dtype=torch.int32), torch.full((B,), n, dtype=torch.int32)
        logits = x.clone()
        ids = sampler.sample_greedy(sampler.GreedyParams(logits=logits, input_lengths=lens, sequence_lengths=lens, token_ids=tokens, step=n, **p))
        return ids.tolist(), logits, tokens

    want, got = run(False), run(True)
    assert got[0] == want[0] and torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    assert built == ([None] if top_k == 5 else [])
