"""Which form tiles_form picks, in calls whose forms were all measured (us on one MI355X): never more than 8 % behind hy_scan, at most a third behind the fastest,
chunks counted with the host time of their launches."""
import pytest

from rtp_llm_amd import hybrid_ops as hops

# rows, sequences, rows of the longest, heads, key channels, value channels; hy_scan, hy_walk whole, in chunks of 32 / 64 / 128
CALLS = [
    (167, 2, 103, 2, 64, 64, dict(scan=39.1, walk=33.9, c32=21.3, c64=31.9)),
    (17, 8, 4, 32, 64, 256, dict(scan=14.8, walk=14.5)),
    (258, 4, 101, 8, 64, 128, dict(scan=39.0, walk=36.0, c32=24.8, c64=35.1)),
    (17, 4, 6, 4, 128, 128, dict(scan=9.3, walk=10.6)),
    (1716, 4, 693, 2, 128, 256, dict(scan=342.6, walk=251.5, c32=39.7, c64=50.8, c128=77.8)),
    (1288, 2, 891, 4, 32, 64, dict(scan=282.8, walk=228.8, c32=25.9, c64=34.4, c128=54.4)),
    (8881, 8, 1658, 4, 64, 64, dict(scan=543.3, walk=441.0, c32=62.4, c64=56.8, c128=76.1)),
    (750, 1, 750, 4, 64, 256, dict(scan=248.2, walk=208.2, c32=31.7, c64=38.1, c128=58.0)),
    (7057, 8, 1342, 8, 96, 128, dict(scan=556.6, walk=475.9, c32=155.5, c64=135.8, c128=123.9)),
    (345, 1, 345, 8, 64, 128, dict(scan=117.7, walk=100.6, c32=25.5, c64=35.0, c128=56.4)),
    (152, 2, 79, 8, 128, 128, dict(scan=44.6, walk=33.0, c32=28.8, c64=44.0)),
    (308, 8, 50, 16, 64, 128, dict(scan=24.9, walk=23.4, c32=35.7)),
    (687, 2, 563, 32, 64, 64, dict(scan=191.7, walk=159.6, c32=43.0, c64=48.2, c128=62.2)),
    (1520, 4, 710, 16, 128, 128, dict(scan=355.1, walk=255.8, c32=95.9, c64=82.2, c128=91.6)),
    (1197, 1, 1197, 8, 64, 128, dict(scan=391.9, walk=329.6, c32=40.2, c64=41.8, c128=60.3)),
    (181, 16, 21, 8, 128, 128, dict(scan=19.0, walk=17.6)),
    (50, 8, 10, 32, 64, 128, dict(scan=13.0, walk=11.7)),
    (144, 1, 144, 4, 64, 256, dict(scan=52.3, walk=44.7, c32=22.8, c64=33.7, c128=56.5)),
    (415, 8, 112, 32, 64, 128, dict(scan=63.2, walk=40.5, c32=51.2, c64=53.5)),
    (5974, 16, 765, 32, 64, 128, dict(scan=677.8, walk=300.3, c32=421.0, c64=314.5, c128=274.1)),
]


@pytest.mark.parametrize("T,nseq,longest,heads,dim,vdim,us", CALLS)
def test_pick(T, nseq, longest, heads, dim, vdim, us):
    C = hops.tiles_form(T, nseq, longest, heads, dim, vdim)
    t = us["scan" if C is None else "walk" if C == 0 else f"c{C}"]
    full = {k: v + hops.CHUNKS_HOST_US * (k[0] == "c") for k, v in us.items()}
    assert t <= 1.08 * us["scan"] and t <= 4 / 3 * min(full.values())
