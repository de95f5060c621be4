"""Which batches of 3 to 255 activation rows the contraction that deals K to wavefronts takes, on the CPU."""
import ctypes

import pytest

from candy_amd import hip, synth

LIB = ctypes.CDLL(hip.LIB_PATH)
LIB.candy_test_rows_i8.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_int] * 5
FORMATS = [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML]


def rule(fmt, rows, cols, m, exact=0, f16_api_min_m=33, i8_min_m=0, small_batch_kernel=1):
    return LIB.candy_test_rows_i8(fmt, rows, cols, m, 256, exact, f16_api_min_m, i8_min_m, small_batch_kernel)


def single(*args, **kw):
    return bool(rule(*args, **kw) & 1)


def prompt(*args, **kw):
    return bool(rule(*args, **kw) & 2)


@pytest.mark.parametrize("fmt", FORMATS)
def test_rows_too_long_for_the_vector_kernels(fmt):
    # 1.3125 bytes a value in 64 KB of LDS: 195 super-blocks; from 16 activation rows on there is no such limit
    for m in (3, 4, 9, 15):
        for exact in (0, 1):
            assert not single(fmt, 4096, 196 * 256, m, exact) and not prompt(fmt, 4096, 196 * 256, m)
    assert prompt(fmt, 4096, 195 * 256, 15) and single(fmt, 4096, 195 * 256, 15)
    assert prompt(fmt, 4096, 196 * 256, 16) and single(fmt, 4096, 65536, 16)


@pytest.mark.parametrize("fmt", FORMATS)
def test_single_contractions_leave_the_batches_that_take_fp16_tiles(fmt):
    k46 = fmt in (synth.Q4_K, synth.Q6_K)
    for option in (16, 20, 33, 64, 65, 100, 1 << 30):
        first = option if k46 else max(option, 65)  # candy_hip.h: the other formats from 65 or this if larger
        for m in (17, 19, 20, 32, 33, 63, 64, 65, 99, 100, 200, 255):
            assert single(fmt, 11000, 4096, m, f16_api_min_m=option) == (m < first), (option, m)
            assert single(fmt, 11000, 4096, m, exact=1, f16_api_min_m=option) and prompt(fmt, 11000, 4096, m, f16_api_min_m=option)


@pytest.mark.parametrize("fmt", FORMATS)
def test_comparison_runs_on_the_vector_kernels(fmt):
    for m in (5, 12, 40):
        assert prompt(fmt, 11000, 4096, m) and prompt(fmt, 11000, 4096, m, i8_min_m=2)
        for kw in (dict(i8_min_m=99), dict(small_batch_kernel=0)):
            assert not prompt(fmt, 11000, 4096, m, **kw) and not single(fmt, 11000, 4096, m, **kw)


def test_q4_k_stays_on_its_one_pass_kernel_up_to_32_super_blocks_a_strip_a_cu():
    for m in (3, 5, 16):
        for rows in (1024, 2048, 4096):
            for blocks, here in ((20, True), (28, True), (29, False), (32, False), (33, True), (43, True)):
                assert single(synth.Q4_K, rows, 256 * blocks, m) == here, (rows, blocks, m)
            assert single(synth.Q4_K, rows - 1, 8192, m)  # rows that kernel does not take
        assert single(synth.Q4_K, 4112, 8192, m) and single(synth.Q5_K, 2048, 8192, m)
    assert single(synth.Q4_K, 2048, 8192, 17) and prompt(synth.Q4_K, 2048, 8192, 16) and single(synth.Q4_K, 2048, 8192, 16, exact=1)


def test_q4_k_stays_on_its_one_pass_kernel_where_the_grid_leaves_slots_idle():
    for m in (3, 8, 16):
        for rows, here in ((16384, False), (16400, False), (24576, False), (30720, True), (32000, True), (40000, False), (48000, True)):
            for cols in (1024, 1536, 4096):
                assert single(synth.Q4_K, rows, cols, m) == here, (rows, cols, m)
            assert single(synth.Q4_K, rows, 4352, m) and single(synth.Q4_K, rows, 512, m) == (rows > 16384)
            assert single(synth.Q4_K, rows, 4096, m, exact=1) == (rows > (16384 if m > 4 else 20000))
        assert single(synth.Q4_K, 64000, 2048, m) == (m > 8)
    assert [single(synth.Q4_K, rows, 2048, 32) for rows in (8192, 12288, 12304, 20000)] == [False, False, True, True]


@pytest.mark.parametrize("fmt", [synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML])
def test_three_and_four_rows_of_the_32_value_formats(fmt):
    for m in (3, 4):
        for rows, cols, here in ((8192, 6144, True), (8208, 6144, False), (16384, 6144, False), (12288, 6400, True),  # two rounds
                                 (16400, 1536, False), (24576, 8192, False), (16400, 14336, False), (40000, 4096, False),  # idle slots
                                 (16400, 1280, True), (30720, 4096, True), (32000, 8192, True), (48000, 4096, True)):
            assert single(fmt, rows, cols, m) == here, (rows, cols, m)
        assert single(fmt, 5000, 4096, m) == (fmt == synth.Q8_0 or m == 4)
        assert single(fmt, 5000, 2048, m) and single(fmt, 5000, 5376, m)
    assert single(fmt, 16400, 4096, 5) and single(synth.Q5_K, 16400, 4096, 3)


# weight rows x values, activation rows: (with one super-block less, with this many)
LEAST = [(synth.Q5_K, 16000, 33, 3), (synth.Q5_K, 32000, 5, 4), (synth.Q5_K, 32000, 33, 7), (synth.Q5_K, 12000, 17, 3), (synth.Q5_K, 8192, 17, 2),
         (synth.Q6_K, 12000, 17, 7), (synth.Q6_K, 20000, 8, 4), (synth.Q6_K, 32000, 8, 6), (synth.Q6_K, 64000, 17, 7), (synth.Q6_K, 64000, 3, 3), (synth.Q6_K, 128000, 4, 6),
         (synth.Q8_0, 8192, 9, 2), (synth.Q8_0, 16000, 17, 2), (synth.Q8_0, 24000, 9, 3), (synth.Q8_0, 24000, 33, 3), (synth.Q4_0, 24000, 33, 4),
         (synth.Q8_0, 32000, 33, 4), (synth.Q4_0, 32000, 33, 6), (synth.Q5_K, 24000, 33, 4)]


@pytest.mark.parametrize("fmt,rows,m,least", LEAST)
def test_rows_of_few_super_blocks(fmt, rows, m, least):
    assert not single(fmt, rows, 256 * (least - 1), m, exact=1) and not prompt(fmt, rows, 256 * (least - 1), m)
    assert prompt(fmt, rows, 256 * least, m) and single(fmt, rows, 256 * least, m, f16_api_min_m=99)


@pytest.mark.parametrize("fmt", FORMATS)
def test_eight_super_blocks_are_enough_and_few_rows_have_no_better_kernel(fmt):
    for rows in (4096, 12000, 64000):
        for m in (3, 5, 12, 20, 60):
            assert prompt(fmt, rows, 2048, m)
    if fmt in (synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML):
        assert single(fmt, 32000, 256, 8) and single(fmt, 32000, 256, 3)


# format, weight rows, values, activation rows: planar quants there, f32 and Q8_0 blocks elsewhere or not
PLANAR = [(synth.Q8_0, 4112, 14336, 3, False), (synth.Q4_0, 4112, 14336, 4, False), (synth.Q8_0, 2048, 4096, 8, False),
          (synth.Q8_0, 4112, 4096, 5, True), (synth.Q8_0, 1024, 8192, 5, True), (synth.Q5_K, 11008, 4096, 3, False),
          (synth.Q5_K, 11008, 4096, 5, True), (synth.Q5_K, 4096, 8192, 3, True), (synth.Q5_K, 1024, 8192, 3, False),
          (synth.Q5_K, 24576, 2048, 3, True), (synth.Q6_K, 4096, 4096, 4, False), (synth.Q6_K, 16384, 2048, 4, False),
          (synth.Q6_K, 11008, 4096, 4, True),
          (synth.Q4_K, 4096, 11008, 3, False), (synth.Q4_K, 4096, 11008, 5, True), (synth.Q4_K, 4096, 14336, 3, True),
          (synth.Q6_K, 11008, 1024, 10, False), (synth.Q5_K, 24576, 1024, 10, False), (synth.Q5_K, 11008, 1024, 10, True),
          (synth.Q5_K, 1024, 2048, 10, False), (synth.Q5_K, 1024, 4096, 10, True), (synth.Q5_K, 2048, 4096, 5, False),
          (synth.Q5_K, 1024, 5120, 5, True), (synth.Q5_K, 4112, 1024, 5, True)]


@pytest.mark.parametrize("fmt,rows,cols,m,here", PLANAR)
def test_planar_quants_where_a_launch_more_pays(fmt, rows, cols, m, here):
    assert single(fmt, rows, cols, m) and single(fmt, rows, cols, m, exact=1) == here


def test_q6_k_tiles_of_more_than_48_rows():
    def shape(rows, m):
        return divmod(LIB.candy_test_rows_q6k_shape(ctypes.c_int64(rows), ctypes.c_int64(m), 256), 100)

    for rows in (16, 1000, 1024, 1536, 2048, 2560, 3072, 5000, 14336, 128256):
        for m in range(49, 256):
            rf, mt = shape(rows, m)
            tiles = -(-m // (16 * mt)) * mt
            assert (rf, mt) in ((2, 4), (1, 4), (1, 3), (1, 2), (1, 1)) and tiles <= (m + 63) // 64 * 4  # the image's tiles
    # a grid that two strips and four tiles would leave half empty takes smaller ones; a full one does not
    assert shape(2048, 100) == (1, 4) and shape(1536, 80) == (1, 1) and shape(3072, 192) == (1, 3)
    assert shape(14336, 255) == (2, 4) and shape(8192, 128) == (2, 4)
