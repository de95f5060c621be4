"""Which tile a contraction on the fp16 tiles takes, on the CPU: the rule for Q4_K rows of up to 16 super-blocks, whose narrow tiles
spare a split of K, and where a prompt leaves them because the launch behind sums the two copies; and rows that are too long for the
role-split tiles' offsets."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth

LIB = ctypes.CDLL(hip.LIB_PATH)


def code(fmt, rows, cols, m, deferred, cus):
    n = len(rows)
    return LIB.candy_test_f16_tile(fmt, (ctypes.c_int64 * n)(*rows), n, ctypes.c_int64(cols), ctypes.c_int64(m), cus, int(deferred))


def tile(rows, cols, m, deferred, cus=256, q4k=True):
    """(weight rows, activation rows)."""
    return divmod(code(synth.Q4_K if q4k else synth.Q8_0, rows, cols, m, deferred, cus), 1000)


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


@pytest.mark.parametrize("m", [65, 128, 129, 300])
def test_rows_of_q8_0_past_32_bit_offsets(m):
    # 128 rows of 17 bytes to 16 values: the last one ends at 2^32 - 1 at the most
    last = (2 ** 32 - 1) // (128 * 272) * 256
    for rows, longest in (((4096,), last), ((200, 128), last), ((127,), (2 ** 32 - 1) // (127 * 272) * 256), ((1,), 2 ** 31 - 256)):
        assert code(synth.Q8_0, rows, longest, m, False, 256) > 0
        if longest < 2 ** 31 - 256:
            assert code(synth.Q8_0, rows, longest + 256, m, False, 256) in (-128128, -128256)
    for fmt in (synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q4_0, synth.Q4_0_GGML):  # through pointers
        assert code(fmt, (4096,), 2 ** 31 - 256, m, False, 256) > 0


def test_gate_and_up_of_q8_0_past_32_bit_offsets():
    # 64 rows of each
    def covers(fmt, cols):
        return LIB.candy_test_f16_silu(fmt, ctypes.c_int64(12288), ctypes.c_int64(cols), ctypes.c_int64(300), 256)

    last = (2 ** 32 - 1) // (64 * 272) * 256
    assert covers(synth.Q8_0, 4096) and covers(synth.Q8_0, last) and not covers(synth.Q8_0, last + 256) and covers(synth.Q4_K, last + 256)


def test_where_the_norm_behind_sums_the_copies():
    # rows that its registers hold, and not behind the last layer's down projection, which no norm of all rows follows: a projection that
    # sums its own copies is no reason for the wide tiles
    behind = LIB.candy_test_norm_sums_behind
    for d_model in (256, 4096, 8192):
        assert all(bool(behind(d_model, 3, layer, down)) == ((layer, down) != (2, 1)) for layer in range(3) for down in (0, 1))
    for d_model in (8448, 11264):
        assert not any(behind(d_model, 3, layer, down) for layer in range(3) for down in (0, 1))
    assert tile((11264,), 1024, 200, False) == (128, 128) and tile((11264,), 1024, 200, True) != (128, 128)


@pytest.mark.parametrize("rows,cols,m,want", [
    # one column of 192-row tiles with K split beside two columns of 128 rows: where those are split too, more than a round, or K is long
    (8192, 2048, 140, (128, 192)), (18432, 2048, 192, (128, 192)), (12288, 2560, 160, (128, 192)), (14336, 3072, 192, (112, 192)), (14336, 2816, 160, (112, 192)),
    (11008, 4096, 140, (128, 192)), (14336, 4096, 180, (112, 192)),
    # a round of whole 128-row tiles, K short: us on 192 / 128 rows 27.0 / 26.3, 29.2 / 26.5, 26.2 / 24.7, 27.8 / 24.9, 25.9 / 24.9, 30.6 / 29.1
    (12288, 2048, 129, (128, 128)), (12288, 2048, 192, (128, 128)), (14336, 2048, 129, (112, 128)), (14336, 2048, 192, (112, 128)),
    (9216, 2048, 192, (128, 128)), (14336, 2560, 192, (112, 128)), (14336, 2816, 192, (112, 128)), (16384, 2304, 192, (128, 128))])
def test_one_column_of_192_rows_or_two_of_128(rows, cols, m, want):
    assert tile((rows,), cols, m, False) == want
