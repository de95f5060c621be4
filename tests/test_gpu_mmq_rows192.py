"""fp16 tiles of 192 activation rows: edges of the tiles and of the padded activation image, whole and split contractions, against
the tiles of 256 rows (the same order of sums along equal splits) and the oracle."""
import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


# 961 rows: six tiles of 192 end past the four of 256; 3584 = 32 x 112 weight rows (Q4_K: tiles of 112)
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML])
@pytest.mark.parametrize("rows,cols,m", [(1030, 4352, 129), (129, 4352, 192), (1030, 4352, 193), (1030, 4352, 300), (130, 4352, 385),
                                         (4099, 512, 961), (3584, 4352, 257)])
def test_tiles_of_192_rows(dev, fmt, rows, cols, m):
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    try:
        for split in (1, 2):
            dev.set_option("mmq.f16_split", split)
            dev.set_option("mmq.f16_shape", 0)
            got = dev.qmatmul(q, x)
            dev.set_option("mmq.f16_shape", 4)  # 128 x 256
            assert np.array_equal(got.view(np.uint32), dev.qmatmul(q, x).view(np.uint32))
    finally:
        dev.set_option("mmq.f16_shape", 0)
        dev.set_option("mmq.f16_split", 0)
    got = dev.qmatmul(q, x)
    sub, some = np.unique(np.r_[0:rows:97, rows - 3:rows]), np.unique(np.r_[0, 15, 16, 47, 48, 127, m - 1])
    want = o.qmatmul(fmt, np.ascontiguousarray(w.reshape(rows, -1)[sub]).reshape(-1), len(sub), cols, x[some])
    # A weight and an activation, each off by at most 2^-11 of itself (2^-11 / sqrt 3 in the mean square), in independent products:
    # sqrt(2 / 3) 2^-11 of the outputs' norm, and 1.7 times that for a norm over as few as 35 of them (their largest value is
    # no scale for the largest error)
    assert np.linalg.norm(got[some][:, sub].astype(np.float64) - want) <= np.sqrt(2) * 2 ** -11 * np.linalg.norm(want)
