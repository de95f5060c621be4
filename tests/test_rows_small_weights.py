"""Weights of few rows keep batches past the fp16 threshold on the exact kernel that deals K to wavefronts, up to a limit."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o

LIB = ctypes.CDLL(hip.LIB_PATH)
LIB.candy_test_rows_i8.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_int] * 5
FORMATS = [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML]


def exact(fmt, rows, cols, m, threshold=33):
    return bool(LIB.candy_test_rows_i8(fmt, rows, cols, m, 256, 0, threshold, 0, 1) & 1)


@pytest.mark.parametrize("fmt", FORMATS)
def test_which_weights_stay(fmt):
    q6k = fmt == synth.Q6_K
    for m in (65, 128, 129, 255):
        assert exact(fmt, 1024, 4096, m) and not exact(fmt, 4097, 4096, m)
        assert exact(fmt, 1024, 2048, m) and not exact(fmt, 1023, 2048, m)  # two million values
        assert not exact(fmt, 1024, 4096, m, threshold=32)
    assert not exact(fmt, 1024, 4096, 256)
    # the work of 1536 x 8192: 1.45 or 2.2 billion products
    assert [exact(fmt, 1536, 8192, m) for m in (115, 116, 174, 175)] == [True, not q6k, not q6k, False]
    assert [exact(fmt, 2048, 8192, m) for m in (86, 87, 119, 120)] == [True, not q6k, not q6k, False]
    assert [exact(fmt, 4096, 2048, m) for m in (129, 244, 245)] == [not q6k, not q6k, False]
    assert exact(fmt, 4096, 1024, 255)
    assert exact(fmt, 4096, 11008, 64) == (fmt not in (synth.Q6_K,)) and not exact(fmt, 4096, 11008, 65)


# the first and the last batch, tiles of 16 rows begun and full, strips of weight rows cut short
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,cols,m", [(1024, 2048, 65), (1001, 2304, 255), (2049, 1024, 240), (4095, 1024, 129), (520, 4352, 97)])
def test_against_the_oracle(fmt, rows, cols, m):
    assert exact(fmt, rows, cols, m)
    w = synth.random_weight(fmt, rows, cols, seed=rows + m)
    x = synth.random_activations(m, cols, seed=cols + m)
    dev = hip.Device(0)
    try:
        got = dev.qmatmul(dev.qtensor(fmt, rows, cols, w), x)
    finally:
        dev.close()
    sub, some = np.unique(np.r_[0:rows:37, rows - 17:rows]), np.unique(np.r_[0, 15, 16, 63, 64, m - 1])
    want = o.qmatmul(fmt, np.ascontiguousarray(w.reshape(rows, -1)[sub]).reshape(-1), len(sub), cols, x[some])
    # exact products summed in f32: 2^-24 of a partial sum at most each, cols of them of random sign
    err = np.linalg.norm(got[some][:, sub].astype(np.float64) - want) / np.linalg.norm(want)
    assert err <= cols ** 0.5 * 2.0 ** -24, err
