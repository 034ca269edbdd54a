"""Which form scan takes on its own, in calls whose forms were all measured (us on one MI355X, on the GPU alone): never more than 10 % behind hy_scan, at most half as much again as the
fastest; a pick without chunks may lose to chunks by the host's time for them.  Constant decays up to FIXED_TILES_FROM rows keep hy_scan whatever it takes."""
import pytest

from rtp_llm_amd import hybrid_ops as hops

# rows, sequences, rows of the longest, heads, key channels, value channels: hy_scan (a constant decay: in chunks where scan_prefers_chunks), hy_walk whole, in chunks of 32 / 64 / 128
GLA, HGRN2, FIXED = hops.SCAN_GLA, hops.SCAN_HGRN2, hops.SCAN_FIXED
CALLS = {
    (167, 2, 103, 2, 64, 64): {GLA: dict(scan=37.6, walk=33.0, c32=21.0, c64=32.8),
                               HGRN2: dict(scan=34.7, walk=32.5, c32=20.5, c64=32.0),
                               FIXED: dict(scan=34.3, walk=28.2, c32=20.0, c64=29.2)},
    (202, 2, 101, 8, 64, 128): {GLA: dict(scan=37.9, walk=34.5, c32=23.1, c64=34.5),
                                HGRN2: dict(scan=34.9, walk=33.9, c32=22.6, c64=33.5),
                                FIXED: dict(scan=34.3, walk=29.5, c32=22.0, c64=30.9)},
    (198, 2, 99, 8, 64, 128): {GLA: dict(scan=37.2, walk=34.6, c32=23.1, c64=34.4),
                               HGRN2: dict(scan=34.3, walk=33.7, c32=22.7, c64=33.5),
                               FIXED: dict(scan=34.0, walk=29.6, c32=22.1, c64=31.1)},
    (8192, 4, 2048, 16, 64, 128): {GLA: dict(scan=678.9, walk=598.1, c32=232.2, c64=171.8, c128=150.3),
                                   HGRN2: dict(scan=609.1, walk=573.0, c32=227.5, c64=171.7, c128=160.3),
                                   FIXED: dict(scan=395.7, walk=443.3, c32=199.2, c64=142.5, c128=132.6)},
    (1537, 1, 1537, 8, 64, 128): {GLA: dict(scan=495.3, walk=437.1, c32=42.3, c64=44.1, c128=64.7),
                                  HGRN2: dict(scan=453.4, walk=432.2, c32=44.5, c64=42.9, c128=62.0),
                                  FIXED: dict(scan=67.5, walk=340.1, c32=42.1, c64=40.2, c128=54.5)},
    (17, 4, 5, 32, 64, 128): {GLA: dict(scan=7.2, walk=8.5),
                              HGRN2: dict(scan=7.1, walk=8.2),
                              FIXED: dict(scan=8.8, walk=9.3)},
    (1560, 8, 195, 8, 128, 256): {GLA: dict(scan=112.5, walk=89.9, c32=96.5, c64=94.8, c128=133.9),
                                  HGRN2: dict(scan=103.1, walk=95.6, c32=102.7, c64=99.9, c128=145.4),
                                  FIXED: dict(scan=99.3, walk=76.2, c32=88.5, c64=85.3, c128=116.6)},
    (11729, 37, 317, 4, 96, 64): {GLA: dict(scan=138.9, walk=134.0, c32=111.8, c64=115.7, c128=128.8),
                                  HGRN2: dict(scan=131.8, walk=143.5, c32=119.9, c64=121.7, c128=140.1),
                                  FIXED: dict(scan=162.0, walk=110.4, c32=99.6, c64=101.0, c128=110.3)},
    (6400, 20, 320, 2, 128, 64): {GLA: dict(scan=160.4, walk=133.8, c32=48.2, c64=54.7, c128=92.5),
                                  HGRN2: dict(scan=152.9, walk=143.1, c32=52.4, c64=57.2, c128=94.9),
                                  FIXED: dict(scan=70.3, walk=110.2, c32=44.9, c64=48.2, c128=77.2)},
    (320, 8, 40, 16, 64, 128): {GLA: dict(scan=19.8, walk=18.1, c32=36.4),
                                HGRN2: dict(scan=18.7, walk=17.5, c32=36.8),
                                FIXED: dict(scan=19.5, walk=16.8, c32=34.3)},
    (1224, 9, 136, 32, 128, 128): {GLA: dict(scan=215.1, walk=86.9, c32=137.7, c64=143.5, c128=154.2),
                                   HGRN2: dict(scan=200.9, walk=101.4, c32=145.4, c64=156.0, c128=167.1),
                                   FIXED: dict(scan=190.0, walk=77.0, c32=125.1, c64=132.5, c128=135.0)},
    (32, 16, 2, 16, 32, 64): {GLA: dict(scan=5.8, walk=7.9),
                              HGRN2: dict(scan=5.8, walk=7.6),
                              FIXED: dict(scan=7.7, walk=8.9)},
    (10232, 8, 1658, 4, 64, 64): {GLA: dict(scan=546.4, walk=477.2, c32=65.3, c64=58.5, c128=80.6),
                                  HGRN2: dict(scan=494.8, walk=454.2, c32=68.1, c64=61.6, c128=83.0),
                                  FIXED: dict(scan=105.0, walk=359.2, c32=58.1, c64=51.6, c128=68.2)},
    (751, 8, 159, 16, 64, 64): {GLA: dict(scan=56.7, walk=47.5, c32=35.1, c64=46.2, c128=60.6),
                                HGRN2: dict(scan=51.9, walk=46.3, c32=36.2, c64=47.5, c128=59.3),
                                FIXED: dict(scan=50.2, walk=39.6, c32=33.2, c64=41.0, c128=51.9)},
    (2814, 2, 1624, 32, 64, 128): {GLA: dict(scan=537.3, walk=478.2, c32=147.7, c64=130.7, c128=116.5),
                                   HGRN2: dict(scan=483.6, walk=454.1, c32=151.2, c64=134.1, c128=122.9)},
    (464, 1, 464, 32, 128, 128): {GLA: dict(scan=231.4, walk=191.5, c32=59.9, c64=76.9, c128=94.5),
                                  HGRN2: dict(scan=219.1, walk=205.8, c32=62.9, c64=82.6, c128=97.4)},
    (17207, 32, 733, 8, 64, 128): {GLA: dict(scan=325.9, walk=217.1, c32=243.1, c64=191.0, c128=194.5),
                                   HGRN2: dict(scan=291.0, walk=205.3, c32=229.9, c64=187.2, c128=195.9)},
    (4672, 4, 1400, 8, 96, 64): {GLA: dict(scan=582.6, walk=575.9, c32=101.8, c64=108.9, c128=125.6),
                                 HGRN2: dict(scan=552.4, walk=612.1, c32=107.8, c64=115.9, c128=135.7)},
    (562, 7, 113, 2, 64, 64): {GLA: dict(scan=41.1, walk=37.2, c32=21.5, c64=33.5),
                               HGRN2: dict(scan=37.9, walk=36.1, c32=21.0, c64=32.2)},
    (906, 8, 171, 16, 64, 128): {GLA: dict(scan=62.4, walk=54.9, c32=47.2, c64=53.1, c128=68.5),
                                 HGRN2: dict(scan=57.6, walk=52.1, c32=48.0, c64=54.2, c128=65.4)},
    (375, 8, 68, 8, 96, 256): {HGRN2: dict(scan=32.4, walk=39.0)},
    (54, 1, 54, 32, 80, 256): {GLA: dict(scan=25.9, walk=29.9)},
    (776, 32, 38, 4, 80, 128): {GLA: dict(scan=20.2, walk=23.5)},
    (5486, 64, 131, 2, 80, 128): {GLA: dict(scan=55.0, walk=61.2)},
    (5840, 32, 282, 4, 128, 256): {GLA: dict(scan=287.8, walk=119.5)},
}


@pytest.mark.parametrize("call", CALLS)
def test_pick(call):
    for mode, us in CALLS[call].items():
        C = hops.scan_form(mode, *call)
        if mode == FIXED and call[2] <= hops.FIXED_TILES_FROM:
            assert C is None
            continue
        t = us["scan" if C is None else "walk" if C == 0 else f"c{C}"]
        host = 0 if C else hops.CHUNKS_HOST_US
        assert t <= 1.1 * us["scan"] and t <= 1.5 * min(v + host * (k[0] == "c") for k, v in us.items()), (mode, C, us)


def test_unknown_longest():
    """max_rows 0: the longest is taken to be what the other sequences leave, a constant decay keeps hy_scan."""
    assert hops.scan_form(FIXED, 4096, 1, 0, 8, 64, 128) is None
    assert hops.scan_form(GLA, 4096, 1, 0, 8, 64, 128) == hops.scan_form(GLA, 4096, 1, 4096, 8, 64, 128)


@pytest.mark.parametrize("call,scan,walk", [((350, 8, 59, 8, 96, 256), 32.2, 38.0), ((171, 4, 65, 8, 64, 64), 26.0, 28.7), ((706, 16, 82, 8, 128, 128), 48.2, 53.4),
                                            ((1815, 16, 176, 16, 128, 192), 267.9, 103.0)])
def test_small_tau(call, scan, walk):
    """Decays of tau 1 cost the tiles more (the last is of tau 16, far from the line)."""
    C = hops.scan_form(GLA, *call, tau=1.0)
    assert C == (0 if walk < scan else None)
