"""Q8_0 on the role-split fp16 tiles, whose blocks come through LDS: one super-block, two and odd numbers of them, ragged tiles, K
split, against the tiles whose lanes load their own runs (the same products in the same order: the same bits)."""
import numpy as np
import pytest

from candy_amd import hip, synth


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


# activation tiles of 128 (at most 128 rows; shape 2), 192 and 256 rows
@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,m,shape", [(129, 256, 128, 2), (2100, 512, 129, 2), (1, 256, 129, 4), (127, 768, 193, 0), (1030, 256, 257, 4),
                                               (2049, 1280, 300, 0), (300, 14336, 512, 4)])
def test_same_bits_as_loads_of_single_lanes(dev, rows, cols, m, shape):
    q = dev.qtensor(synth.Q8_0, rows, cols, synth.random_weight(synth.Q8_0, rows, cols, seed=rows + cols))
    x = synth.random_activations(m, cols, seed=m)
    try:
        for split in (1, 2):
            dev.set_option("mmq.f16_split", split)
            dev.set_option("mmq.f16_shape", shape)
            got = dev.qmatmul(q, x)
            dev.set_option("mmq.f16_shape", 3)
            assert np.array_equal(got.view(np.uint32), dev.qmatmul(q, x).view(np.uint32))
    finally:
        dev.set_option("mmq.f16_shape", 0)
        dev.set_option("mmq.f16_split", 0)
