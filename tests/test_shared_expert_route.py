"""Which steps run a mixture's shared expert in the grouped linears of the others: decided on the host."""
import pytest
import torch

from rtp_llm_amd import mixers


class _Asked(Exception):
    pass


def _mixture(W, ff, E, dtype=torch.bfloat16, seed=0, shared=None):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    shared = shared or mixers.GatedMLP(r(ff, W), r(ff, W), r(W, ff), act="silu")
    return mixers.RoutedExperts(mixers.RouterSpec(E, 2), r(E, W), [r(ff, W) for _ in range(E)], [r(ff, W) for _ in range(E)], [r(W, ff) for _ in range(E)], shared, act="silu")


def _asks(monkeypatch, m, T):
    """Whether a forward pass over T rows asks the sort for the shared expert's rows."""
    def sort(*a, shared=False, **k):
        raise _Asked(bool(shared))
    monkeypatch.setattr(mixers.hops, "moe_route_sorted", sort)
    W, E = m.w_down.shape[1], m.router.experts
    with pytest.raises(_Asked) as e:
        m.forward(torch.zeros(1, W, dtype=m.w_down.dtype).expand(T, W), torch.zeros(1, E).expand(T, E))
    return e.value.args[0]


# 65 rows and more, up to 12e9 products of a linear: above them the shared expert's own launches have larger tiles (fp32 has one)
@pytest.mark.parametrize("W,ff,last", [(1024, 704, 16645), (256, 96, 488281), (2048, 2048, 2861)])
def test_many_rows_of_a_large_expert_run_alone(monkeypatch, W, ff, last):
    m = _mixture(W, ff, 2)
    assert [_asks(monkeypatch, m, T) for T in (1, 64, 65, last, last + 1, 4 * last)] == [False, False, True, True, False, False]
    if W == 1024:
        assert _asks(monkeypatch, _mixture(W, ff, 2, torch.float32), 4 * last)


class _Other:
    """A shared expert of a kind of its own: nothing but forward."""

    def forward(self, h):
        return h.float()


def test_a_shared_expert_of_another_kind_runs_alone(monkeypatch):
    class Wrapped(mixers.GatedMLP):
        def forward(self, h):
            return super().forward(h) * 2

    r = lambda *s: torch.randn(*s).bfloat16()
    wrapped = Wrapped(r(96, 256), r(96, 256), r(256, 96), act="silu")
    before = wrapped.w_gate_up, wrapped.w_down
    poly = mixers.PolyNormMLP(r(96, 256), r(256, 96), torch.ones(4), 1e-6)
    for shared in (_Other(), poly, wrapped):
        assert not _asks(monkeypatch, _mixture(256, 96, 2, shared=shared), 100)
    assert wrapped.w_gate_up is before[0] and wrapped.w_down is before[1]


@pytest.mark.parametrize("what", ["shared gate and up", "shared down", "shared in place", "gate and up", "down", "activation", "parameter", "none", "another"])
def test_weights_given_later_are_the_ones_that_run(monkeypatch, what):
    """The stack of all weights stands for the attributes only while they are parts of it."""
    m, other = _mixture(256, 96, 3), _mixture(256, 96, 3, seed=1)
    assert _asks(monkeypatch, m, 100)
    if what == "shared gate and up":
        m.shared.w_gate_up = other.shared.w_gate_up.clone()
    elif what == "shared down":
        m.shared.w_down = other.shared.w_down.clone()
    elif what == "shared in place":                                  # a copy into the view reaches the stack
        m.shared.w_down.copy_(other.shared.w_down)
        assert torch.equal(m.w_all[1][3], other.shared.w_down) and _asks(monkeypatch, m, 100)
        return
    elif what == "gate and up":
        m.w_gate_up = other.w_gate_up.clone()
    elif what == "down":
        m.w_down = other.w_down.clone()
    elif what == "activation":
        m.shared.act = mixers.hops.ACT_RELU
    elif what == "parameter":
        m.shared.act_param = 1.0
    elif what == "none":
        m.shared = None
    elif what == "another":
        m.shared = other.shared
    assert not _asks(monkeypatch, m, 100)
