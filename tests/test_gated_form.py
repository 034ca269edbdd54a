"""What gated_form answers, against the times that it was fitted to: those of a walk token by token (us on one MI355X).  The pick costs no more than hy_scan, and at most a third more than
the fastest (the model's own error).  What hy_walk's tiles take, and the rule in use, is in test_scan_form.py."""
import pytest

from rtp_llm_amd import hybrid_ops as hops

# rows, sequences, rows of the longest, heads, key channels, value channels; hy_scan, hy_walk whole, in chunks of 32 / 64 / 128
CALLS = [
    (1560, 8, 195, 8, 128, 256, dict(scan=104.9, walk=137.0, c32=197.1, c64=180.9, c128=249.3)),
    (11729, 37, 317, 4, 96, 64, dict(scan=141.3, walk=237.4, c32=308.0, c64=286.2, c128=356.5)),
    (630, 18, 35, 16, 32, 64, dict(scan=18.1, walk=22.7, c32=53.2)),
    (70, 10, 7, 32, 64, 64, dict(scan=9.3, walk=10.2)),
    (3542, 11, 322, 4, 128, 256, dict(scan=170.5, walk=234.0, c32=219.8, c64=209.3, c128=276.5)),
    (195, 15, 13, 16, 64, 64, dict(scan=10.0, walk=10.9)),
    (4400, 20, 220, 4, 128, 128, dict(scan=113.9, walk=149.8, c32=150.0, c64=168.9, c128=164.7)),
    (2535, 13, 195, 16, 64, 64, dict(scan=68.5, walk=80.5, c32=86.7, c64=91.0, c128=105.6)),
    (32, 16, 2, 16, 32, 64, dict(scan=5.9, walk=6.6)),
    (1224, 9, 136, 32, 128, 128, dict(scan=207.5, walk=330.9)),
    (1160, 2, 833, 32, 96, 128, dict(scan=333.6, walk=534.3, c32=239.4, c64=252.5, c128=309.7)),
    (1208, 7, 581, 16, 128, 128, dict(scan=272.9, walk=377.5, c32=156.2, c64=177.5, c128=173.0)),
    (12155, 42, 1913, 8, 64, 64, dict(scan=573.0, walk=721.1, c32=187.9, c64=177.8, c128=191.9)),
    (739, 1, 739, 2, 128, 128, dict(scan=361.6, walk=521.1, c32=60.9, c64=97.3, c128=175.3)),
    (2051, 7, 1862, 4, 32, 256, dict(scan=583.4, walk=803.2, c32=73.1, c64=72.4, c128=108.4)),
    (10275, 15, 685, 16, 96, 64, dict(scan=303.9, walk=506.9)),
    (2425, 26, 602, 32, 128, 64, dict(scan=413.1, walk=575.4)),
    (3839, 22, 506, 32, 128, 128, dict(scan=825.9, walk=648.0)),
    (225, 25, 9, 8, 64, 256, dict(scan=17.0, walk=11.9)),
    (8192, 4, 2048, 16, 64, 128, dict(scan=684.0, walk=683.0, c128=265.0)),
]


@pytest.mark.parametrize("T,nseq,longest,heads,dim,vdim,us", CALLS)
def test_pick(T, nseq, longest, heads, dim, vdim, us):
    C = hops.gated_form(T, nseq, longest, heads, dim, vdim)
    t = us["scan" if C is None else "walk" if C == 0 else f"c{C}"]
    assert t <= us["scan"] and t <= 4 / 3 * min(us.values())
