"""Grids of 128 x 256 fp16 tiles whose last round of workgroups is nearly empty take 128 x 128 tiles: against the oracle and
against the wider tiles, whose sums along the contraction have the same order."""
import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML])
@pytest.mark.parametrize("rows,cols,m", [(11008, 512, 513), (10900, 256, 640), (10881, 1024, 577), (10881, 256, 641)])
def test_narrow_tiles_where_they_take_no_more_rounds(dev, fmt, rows, cols, m):
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    got = dev.qmatmul(q, x)
    dev.set_option("mmq.f16_shape", 4)  # 128 x 256 tiles
    try:
        wide = dev.qmatmul(q, x)
    finally:
        dev.set_option("mmq.f16_shape", 0)
    assert np.array_equal(got.view(np.uint32), wide.view(np.uint32))
    sub, some = np.unique(np.r_[0:rows:211, rows - 130:rows]), np.unique(np.r_[0, 127, 128, 255, 256, 511, 512, m - 1])
    want = o.qmatmul(fmt, np.ascontiguousarray(w.reshape(rows, -1)[sub]).reshape(-1), len(sub), cols, x[some])
    # weights and activations rounded to fp16 (2^-11 each), exact products, f32 sums
    assert np.max(np.abs(got[some][:, sub] - want)) <= 5e-4 * np.max(np.abs(want))
