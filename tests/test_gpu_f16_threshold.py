"""mmq.f16_api_min_m: from this many rows a single contraction runs on fp16 tiles, below it every product is exact."""
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
@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q6_K, synth.Q8_0])
def test_the_threshold_is_the_option(dev, fmt):
    rows, cols = 4099, 512
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    q = dev.qtensor(fmt, rows, cols, w)
    others = fmt not in (synth.Q4_K, synth.Q6_K)
    for first, m in ((16, 20), (16, 70), (33, 32), (33, 33), (100, 70), (100, 100), (1 << 20, 130)):
        x = synth.random_activations(m, cols, seed=m)
        dev.set_option("mmq.f16_api_min_m", first)
        try:
            got = dev.qmatmul(q, x)
        finally:
            dev.set_option("mmq.f16_api_min_m", 33)
        sub = np.unique(np.r_[0, m // 2, m - 1])
        want = o.qmatmul(fmt, w, rows, cols, x[sub])
        err = np.linalg.norm(got[sub].astype(np.float64) - want) / np.linalg.norm(want)
        # f32 sums of exact products are within 1e-6; operands rounded to fp16 (2^-11 each) come to more than 1e-4
        assert (err > 5e-5) == (m >= (max(first, 65) if others else first)), (first, m, err)
        assert err < 2.0 ** -10
