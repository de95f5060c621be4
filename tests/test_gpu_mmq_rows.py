"""fp16 contraction of up to 128 activation rows with K dealt to the wavefronts, against the 128 x 128 tiles on the same fp16
operands and against the oracle."""
import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


# activation rows at the edges of their fragments (and 129: the tiles); weight rows that fill one, two and three fragments
# per workgroup, one row over each, and one over what a round of workgroups takes; fewer super-blocks than wavefronts, as
# many, and one more; a row length not in fours of weight rows
SHAPES = [(65, 2048, 256), (80, 2049, 2304), (81, 4097, 512), (96, 8193, 768), (97, 2051, 2048), (128, 6000, 1024), (129, 2048, 512),
          (77, 12288, 512), (70, 12289, 256), (66, 2050, 4096)]


@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML])
@pytest.mark.parametrize("m,rows,cols", SHAPES + [(33, 2048, 512), (48, 4100, 2048), (49, 2303, 768), (64, 2048, 1280)])
def test_rows_against_tiles_and_oracle(dev, fmt, m, rows, cols):
    w = synth.random_weight(fmt, rows, cols, seed=rows + m)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    got = dev.qmatmul(q, x)
    assert np.array_equal(got.view(np.uint32), dev.qmatmul(q, x).view(np.uint32))
    dev.set_option("mmq.f16_shape", 2)
    try:
        tiles = dev.qmatmul(q, x)
    finally:
        dev.set_option("mmq.f16_shape", 0)
    top = np.max(np.abs(tiles))
    # the same products in another order: K sums of f32, 2^-24 each of a partial sum no larger than the largest result's
    # order (random signs: sqrt(K) of them, 64 * 2^-24 = 4e-6 at K = 4096)
    assert np.max(np.abs(got - tiles)) <= 4e-6 * top
    sub = np.unique(np.r_[0:rows:97, rows - 17:rows])
    nb = synth.weight_nbytes(fmt, 1, cols)
    want = o.qmatmul(fmt, w.reshape(rows, nb)[sub].reshape(-1), len(sub), cols, x)
    # fp16 operands: 2^-12 of each product, as for the tiles
    assert np.max(np.abs(got[:, sub] - want)) <= 5e-4 * np.max(np.abs(want))
