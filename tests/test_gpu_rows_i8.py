"""The exact contraction of 3 to 255 activation rows with K dealt to wavefronts: every tile shape and its edges, against the
oracle, the int8 tile and vector kernels (other order of f32 sums) and between the entry points."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o

FORMATS = [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML]
# Weight rows (off the strips of 16 and off the float4 stores), values per row (one super-block; fewer than, as many as and one
# more than the wavefronts), activation rows on both sides of every tile's edge; one, two and four strips per workgroup.
SHAPES = [(4099, 256, m) for m in (5, 16, 33, 64)] + [(1030, 1024, m) for m in (5, 17, 48, 49, 255)] + \
         [(258, 4352, m) for m in (16, 17, 65)] + [(2052, 2304, m) for m in (17, 32, 48, 64, 130)] + \
         [(4096, 4096, 18), (16500, 256, 7), (12500, 256, 31), (16500, 256, 40), (16500, 256, 50), (5000, 1024, 3)]


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def rel_err(got, want):
    return float(np.max(np.abs(got.astype(np.float64) - want)) / np.max(np.abs(want)))


def exact(dev, w, x):
    """candy_hip_qmatmul_qact: the exact kernels up to 255 rows."""
    L, act = hip.lib(), ctypes.c_void_p()
    m, cols = x.shape
    src, dst = dev.alloc(x.nbytes), dev.alloc(4 * m * w.rows)
    src.upload(x)
    hip._check(L.candy_hip_qact_create(dev.handle, m, cols, ctypes.byref(act)))
    hip._check(L.candy_hip_qact_quantize(act, src.ptr, m, cols))
    hip._check(L.candy_hip_qmatmul_qact(dev.handle, w.handle, act, dst.ptr))
    out = dst.download(np.float32, m * w.rows).reshape(m, w.rows)
    hip._check(L.candy_hip_qact_free(act))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,cols,m", SHAPES)
def test_rows_against_oracle_and_other_kernels(dev, fmt, rows, cols, m):
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    got = exact(dev, q, x)
    assert np.array_equal(got.view(np.uint32), exact(dev, q, x).view(np.uint32))
    dev.set_option("rows.i8", 0)
    try:
        other = exact(dev, q, x)
    finally:
        dev.set_option("rows.i8", 1)
    # exact integer dots of 32 values; K / 32 products of two scales and their sum in f32, in two orders
    assert rel_err(got, other) <= 2e-6
    sub = np.arange(m) if m <= 16 else np.unique(np.r_[0, 15, 16, m // 2, m - 1])
    want = o.qmatmul(fmt, w, rows, cols, x[sub])
    assert rel_err(got[sub], want) <= 2e-5
    if m <= 16:  # f32 rows and Q8_0 blocks go through other kernels into the same operands
        assert np.array_equal(dev.qmatmul(q, x).view(np.uint32), dev.qmatmul_q8(q, dev.quantize_q8_0(x), m).view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [synth.Q8_0, synth.Q6_K])
def test_a_row_reaches_its_own_results_only(dev, fmt):
    # the image of 5 rows is a tile of 16: what earlier calls left in the other rows, here infinities, must not be seen
    w = synth.random_weight(fmt, 4096, 512, seed=3)
    q = dev.qtensor(fmt, 4096, 512, w)
    x = synth.random_activations(16, 512, seed=4)
    want = dev.qmatmul(q, x[:5])
    x[5:] = np.inf
    dev.qmatmul(q, x)
    exact(dev, q, x)
    assert np.array_equal(dev.qmatmul(q, x[:5]).view(np.uint32), want.view(np.uint32))
    assert np.array_equal(exact(dev, q, x[:5]).view(np.uint32), exact(dev, q, x[:5]).view(np.uint32))
    assert np.all(np.isfinite(exact(dev, q, x[:5])))
