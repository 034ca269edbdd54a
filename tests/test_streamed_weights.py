"""Which models' weights are read past the memory-side cache: those of which a step reads more than it holds."""
import torch

import dupenex_util as U
from rtp_llm_amd import hybrid_ops as hops
from rtp_llm_amd.hybrid import HybridConfig, HybridModel


def test_by_the_bytes_of_a_step():
    class Other:
        pass

    a, b, c = torch.zeros(4), torch.zeros(2), Other()
    c.t = torch.zeros(3)
    assert not hops.mark_streamed([a, {"b": b}], 100, 100) and not hasattr(a, "streamed")
    assert hops.mark_streamed([a, {"b": (b, None)}, c, 7], 101, 100) and a.streamed and b.streamed and not hasattr(c.t, "streamed")      # objects of other packages are not looked into


def test_model_weights(monkeypatch):
    seen, mark = [], hops.mark_streamed
    monkeypatch.setattr(hops, "mark_streamed", lambda w, nbytes: seen.append(nbytes) or mark(w, nbytes, nbytes - 1 if len(seen) > 1 else nbytes))
    cfg = U.make_config([U.parallel_layer(mlp=U.moe()), U.delta_layer()])
    w = U.make_weights(cfg)
    for marked in (False, True):
        m = HybridModel(HybridConfig.from_json(cfg), w, torch.float32, "cpu")
        mats = [m.head, m.layers[0][1].left.w_o, m.layers[0][2].w_gate_up, m.layers[1][1].w_o]
        assert [getattr(t, "streamed", False) for t in mats] == [marked] * 4
    embed = 0 if m.cfg.tied_head else w["embed"].numel() * 4
    assert seen[0] == seen[1] <= sum(t.numel() * 4 for t in w.values()) - embed and seen[0] > 0.8 * (sum(t.numel() * 4 for t in w.values()) - embed)
