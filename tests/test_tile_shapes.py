"""The lists of the tile tests reach every tile shape that a call can take: the shape chosen for each listed call, against all shapes chosen over a grid of sizes."""
import pytest
import test_gpu_dense_lean_epilogue as lean
import test_gpu_dense_tiles as dense
import test_gpu_prefill_gemm as prefill
import test_gpu_prefill_stores as stores

from rtp_llm_amd import _C


def _prefill(M, K, N, bf16, wbits):
    """The tile shape of a call that runs one, None for two in one launch."""
    args = (M, -(-N // 16), -(-K // 128), bf16, wbits)
    return None if _C.lib().mi355_gemm_prefill_rest(*args, 128, 1) else _C.lib().mi355_gemm_prefill_shape(*args)


@pytest.mark.parametrize("wbits", [4, 8, 16])
@pytest.mark.parametrize("bf16", [0, 1])
def test_prefill_shapes(bf16, wbits):
    can = {_prefill(M, K, N, bf16, wbits) for M in (65, 96, 129, 200, 257, 300, 513, 1024, 1537, 2050, 3000, 4096, 8192) for K in (128, 256, 384, 640, 896, 1280, 3584, 4864, 18944)
           for N in (24, 64, 200, 512, 1152, 3584, 4608, 9728, 18944, 37888, 151936)}
    can.discard(None)
    assert len(can) >= 5
    assert {_prefill(M, K, N, bf16, wbits) for M, K, N in prefill.SHAPES} - {None} == can


@pytest.mark.parametrize("cols", [1, 2, 7, 8, 14, 43, 72, 74])
@pytest.mark.parametrize("rows", [1, 2, 7, 8, 9, 16, 17, 25, 65])
def test_prefill_tiles_once(rows, cols):
    """Whatever the order in which the blocks take the tiles: each tile once; the blocks of an XCD take a run of whole columns of at most 8 row tiles."""
    tile = _C.lib().mi355_gemm_prefill_tile
    got = [(t & 0xffffffff, t >> 32) for t in (tile(i, rows, cols) for i in range(rows * cols))]
    assert sorted(got) == [(c, r) for c in range(cols) for r in range(rows)]
    if cols % 8 == 0:
        assert got == [(c, r) for r in range(rows) for c in range(cols)]
    elif rows <= 8:
        run = [t for x in range(8) for t in got[x::8]]
        assert run == [(c, r) for c in range(cols) for r in range(rows)]


def test_dense_shapes():
    pick = _C.hybrid_lib().mi355_dense_tile_shape
    can = {pick(M, N, K, 1, 0) for M in (17, 65, 300, 768, 1537, 2304, 4700, 6000, 8190) for N in (8, 200, 1032, 2044, 4100, 16400) for K in (8, 40, 136, 264, 1032, 2056)}
    assert can == {0, 1, 2, 3, 4}
    assert {pick(M, N, K, 1, 0) for M, N, K in dense.SHAPES} == can
    # gated calls: the small tile, both middle ones that they are given in practice, the largest
    assert {0, 1, 4} <= {pick(M, N, K, 1, 0) for M, N, K in dense.GATED}
    # the largest tile with an even and an odd count of K tiles of 32, both with a remainder
    assert {K // 32 % 2 for M, N, K in dense.SHAPES if pick(M, N, K, 1, 0) == 4 and K % 32} == {0, 1}
    assert {pick(M, N, K, 1, 64) for M, N, K in dense.SHAPES} <= {0, 1, 2}           # sorted rows: tiles of 64


def test_dense_lean_store_shapes():
    pick = _C.hybrid_lib().mi355_dense_tile_shape
    assert {pick(M, N, K, 1, 0) for M, N, K in lean.SIZES} == {pick(M, N - 3, K, 1, 0) for M, N, K in lean.SIZES} == {0, 1, 2, 3, 4}
    assert {pick(M, dv, R, H, 0) for M, H, R, dv in lean.HEADS} == {0, 1, 2, 3, 4}


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("kind,group", stores.KINDS)
def test_prefill_store_shapes(kind, group, bf16):
    """Each tile whose results pass through LDS, by class: a launch of that shape alone, a last tile of some rows and one of some columns, gated rows of whole 16 bytes."""
    bits = {"w4": 4, "int8": 8, "fp16": 16}[kind]
    tile = {0: (128, 512), 1: (128, 256), 2: (64, 256)}
    seen = set()
    for M, K, N in stores.SHAPES:
        args = (M, -(-N // 16), K // 128, bf16, bits, group, 1)
        s = _C.lib().mi355_gemm_prefill_form(*args) & 15
        if s in tile and not _C.lib().mi355_gemm_prefill_rest(*args) and M % tile[s][0] and N % tile[s][1] and N % 16 == 0:
            seen.add(s)
    assert seen >= {1, 2} | ({0} if not bf16 and kind != "fp16" and group != 32 else set())
