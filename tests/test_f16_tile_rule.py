"""Which tile a contraction on the fp16 tiles takes, on the CPU: the rule for Q4_K rows of up to 16 super-blocks, whose narrow tiles
spare a split of K, and where a prompt leaves them because the launch behind sums the two copies."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip

LIB = ctypes.CDLL(hip.LIB_PATH)


def tile(rows, cols, m, deferred, cus=256, q4k=True):
    """(weight rows, activation rows)."""
    n = len(rows)
    return divmod(LIB.candy_test_f16_tile(int(q4k), (ctypes.c_int64 * n)(*rows), n, ctypes.c_int64(cols), ctypes.c_int64(m), cus, int(deferred)), 1000)


def wide_split(rows, cols, m, cus=256):
    """Workgroups that share a 128 x 256 tile's K."""
    tiles = sum(-(-r // 128) for r in rows) * -(-m // 256)
    return max(1, min(cus // tiles, cols // 512, 16)) if tiles < 3 * cus // 4 else 1


QKV_8B, O_8B, QKV_1B, O_1B = (4096, 1024, 1024), (4096,), (2048, 512, 512), (2048,)


@pytest.mark.parametrize("rows,cols,m,want", [
    # two copies for the launch behind: us of an 8B-shaped prompt, four layers and the head, narrow / wide: 300 tokens 1179 / 1143, 512 1381 / 1367
    (QKV_8B, 4096, 300, (128, 192)), (QKV_8B, 4096, 512, (128, 256)), (O_8B, 4096, 513, (128, 192)), (O_8B, 4096, 1024, (128, 256)),
    (O_1B, 2048, 1500, (128, 192)),
    # not split on either tile: 240 workgroups of the narrow one are a whole round, 144 of the wide one are not (520 tokens 1608 / 1621,
    # 577 1804 / 1830, 640 1815 / 1835)
    (QKV_8B, 4096, 513, (128, 128)), (QKV_8B, 4096, 576, (128, 128)), (QKV_8B, 4096, 577, (128, 128)), (QKV_8B, 4096, 640, (128, 128)),
    # too few super-blocks to split
    (O_1B, 512, 1024, (128, 128)), (O_8B, 768, 512, (128, 128)),
    # more than two copies
    (O_8B, 4096, 512, (128, 128)), (QKV_1B, 2048, 512, (128, 128)),
])
def test_wide_tiles_where_two_copies_are_left_for_the_launch_behind(rows, cols, m, want):
    assert tile(rows, cols, m, True) == want
    narrow = tile(rows, cols, m, False)
    assert narrow == (128, 128)


def test_nothing_but_two_copies_moves_a_call():
    rng = np.random.default_rng(11)
    moved = 0
    for _ in range(20000):
        rows = [int(rng.integers(1, 100)) * 128 for _ in range(rng.integers(1, 4))]
        cols, m, cus, q4k = 256 * int(rng.integers(1, 40)), int(rng.integers(1, 2100)), int(rng.choice([64, 256, 304])), rng.random() < 0.8
        alone, behind = tile(rows, cols, m, False, cus, q4k), tile(rows, cols, m, True, cus, q4k)
        if alone != behind:
            moved += 1
            assert q4k and cols <= 4096 and m > 128 and alone[1] == 128 and wide_split(rows, cols, m, cus) == 2
        assert q4k or alone[0] == 128
    assert moved > 100
