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
