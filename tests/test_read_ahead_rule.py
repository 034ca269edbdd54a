"""Which weights of a mixture are read ahead of their grouped linears, in layers that were timed both ways (us of the sort and both linears on one MI355X, weights from memory): none that
loses more than 3 % by it, and the ones that gain most."""
import pytest

from rtp_llm_amd.mixers import ahead_from

MB = 1 << 20
# pairs, experts, MB of the gate and up weights (the down weights are half), us without / with
LAYERS = [(71, 8, 40, 32.0, 40.4), (131 * 2, 16, 82, 48.0, 56.9), (186, 8, 36, 31.1, 33.5), (260, 32, 40, 34.3, 39.4), (347, 4, 37, 41.4, 46.7), (364, 64, 96, 49.7, 66.7), (479, 2, 3, 21.8, 25.0),
          (1148, 8, 144, 119.0, 127.1), (1690, 4, 5, 28.0, 29.8), (2507, 4, 1.5, 22.9, 23.4), (4365, 2, 39, 219.3, 195.3), (5318, 4, 7.5, 59.4, 51.9), (6148, 16, 44, 85.8, 73.6),
          (8192, 32, 136, 146.5, 152.2), (12796, 8, 11, 88.4, 82.2), (17216, 16, 24, 144.0, 124.2), (27896, 16, 24, 176.1, 156.7)]


@pytest.mark.parametrize("pairs,experts,mb,off,on", LAYERS)
def test_read_ahead_rule(pairs, experts, mb, off, on):
    takes = pairs >= ahead_from(experts, int(mb * MB)), pairs >= ahead_from(experts, int(mb * MB / 2))
    if on > 1.03 * off:
        assert not takes[0] and (not takes[1] or mb > 96)
    if on < 0.95 * off and pairs >= 4096:
        assert takes == (True, True)


def test_read_ahead_edges():
    assert ahead_from(16, 2 * MB) == 4096 and ahead_from(1025, 48 * MB) == 4100
    assert ahead_from(16, 2 * MB - 1) == ahead_from(16, 48 * MB + 1) == float("inf")
