"""The rules that choose the tile of a bfloat16 contraction, on the CPU: a tile's loads address it through 32-bit byte offsets
(every one of its rows has to lie within 4 GB), no tile of block-diagonal weights reaches into a second block, and the copies of
a contraction in front of a router go by the shape alone."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip

LIB = ctypes.CDLL(hip.LIB_PATH)
LIB.candy_test_dense_plan.argtypes = [ctypes.c_int] * 2 + [ctypes.c_int64] * 3 + [ctypes.c_int] * 4 + [ctypes.POINTER(ctypes.c_int)]
LIB.candy_test_dense_plan.restype = None
LIB.candy_test_grouped_tile_rows.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64]
LIB.candy_test_grouped_weight_rows.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64, ctypes.c_int]
LIMIT = 1 << 32
TILES = {(256, 256), (224, 256), (192, 256), (160, 256), (128, 256), (256, 128), (192, 128), (128, 128)}


def plan(m, rows, ld, ldx=None, partial=0, steady=0, few=0, block_rows=0):
    out = (ctypes.c_int * 4)()
    LIB.candy_test_dense_plan(256, m, rows, ld, ld if ldx is None else ldx, partial, steady, few, block_rows, out)
    return list(out)


def pad64(n):
    return (n + 63) // 64 * 64


@pytest.mark.parametrize("few,partial,steady", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 1, 1)])
def test_offsets_of_a_tile_fit_32_bits(few, partial, steady):
    rng = np.random.default_rng(few + 2 * partial + 4 * steady)
    lds = [64, 4096, 1 << 22, (1 << 23) - 64, 1 << 23, (1 << 23) + 64, 1 << 24, (1 << 24) + 64, 1 << 27, 0x7FFFFFC0]
    for ld in lds:
        for ldx in {ld, min(2 * ld, 0x7FFFFFC0), max(ld, 1 << 25)}:
            for _ in range(20):
                m, rows = int(2 ** rng.uniform(6.1, 14)), pad64(int(2 ** rng.uniform(0, 15)))
                big, bn, bm, splits = plan(m, rows, ld, ldx, partial, steady, few)
                assert 1 <= splits <= 8
                if big:
                    assert (bn, bm) in TILES and (not few or bn in (128, 256))
                    assert bn * ld * 2 <= LIMIT - 1 and bm * ldx * 2 <= LIMIT - 1, (m, rows, ld, ldx, bn, bm)
                else:
                    assert (bn, bm) == (128, 64)
                    assert 128 * max(ld, ldx) * 2 > LIMIT - 1  # only where no large tile can


def test_large_tiles_where_they_were():
    for m in (65, 300, 2000):
        for rows, ld in ((64, 64), (4096, 4096), (14336, 4096), (4096, 14336)):
            assert plan(m, rows, ld)[0] == 1
    assert plan(64, 4096, 4096)[0] == 0


@pytest.mark.parametrize("block_rows", [128, 256, 384, 640])
def test_blocks_are_whole_tiles(block_rows):
    for m in (65, 200, 3000):
        for few in (0, 1):
            big, bn, bm, _ = plan(m, block_rows * 7, block_rows, block_rows * 7, few=few, block_rows=block_rows)
            assert big and block_rows % bn == 0 and (bn, bm) in TILES


def test_copies_in_front_of_a_router_go_by_the_shape():
    for m in (65, 128, 129, 400, 2048):
        for rows in (64, 1600, 2048, 3072, 5120):
            for ld in (320, 1024, 2816, 4096):
                room = 512 // (-(-m // 128) * -(-rows // 128))
                assert plan(m, rows, ld, partial=1, steady=1)[3] == max(1, min(room, 8, ld // 512)), (m, rows, ld)


def test_grouped_tiles_fit_32_bits():
    for experts in (1, 16, 64):
        for slots in (95 * experts, 96 * experts, 1 << 16):
            for widest in (64, 4096, 1 << 22, (1 << 23) - 64, 1 << 23, 1 << 25):
                rows = LIB.candy_test_grouped_tile_rows(experts, slots, widest)
                assert rows in (64, 128)
                if rows == 128:  # 256 weight rows beside them
                    assert slots * widest * 2 <= LIMIT - 1 and 256 * widest * 2 <= LIMIT - 1


# (experts, rows of each, width, rows of an expert's weight) -> rows of a tile, its weight rows: short contractions, few tiles, many
@pytest.mark.parametrize("experts,rows,d,ff,tile,wide", [
    (64, 95, 2048, 1408, 64, None), (64, 96, 2048, 1408, 128, 256), (64, 192, 2048, 1408, 128, 256), (64, 256, 512, 256, 64, None),
    (64, 112, 1024, 512, 64, None), (64, 192, 1024, 512, 128, 256), (8, 96, 4096, 4096, 128, 128), (8, 128, 4096, 4096, 128, 256),
    (4, 256, 1024, 2048, 128, 128), (16, 192, 4096, 2048, 128, 256), (200, 1000, 1088, 128, 128, 128)])
def test_tiles_of_rows_dealt_to_experts(experts, rows, d, ff, tile, wide):
    assert LIB.candy_test_grouped_tile_rows(experts, experts * rows, max(d, ff)) == tile
    if wide:
        assert LIB.candy_test_grouped_weight_rows(256, experts, experts * rows, ff) == wide


def test_narrow_tiles_where_their_last_column_is_half_full():
    def pays(m, rows, ld):
        return bool(LIB.candy_test_narrow_pays(256, *(ctypes.c_int64(v) for v in (m, rows, ld))))

    for m in (2, 32, 33, 64):
        assert pays(m, 8192, 8192) and pays(m, 16384, 8192) and not pays(m, 16448, 8192)
    assert [m for m in range(65, 129) if pays(m, 8192, 8192)] == list(range(97, 129))  # two columns: 512 workgroups
    assert all(pays(m, 8192, 1536) for m in range(65, 129)) and all(pays(m, 7168, 8192) for m in range(65, 129))
    assert not any(pays(m, 8256, 1536) for m in range(65, 129))
