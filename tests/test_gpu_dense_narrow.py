"""The narrow tiles of bfloat16 contractions (32 weight rows, five stages of K in flight): fewer, as many and more stages than fit,
rows on both sides of a tile's edge, against f64 and, bit for bit, against the other tiles' order of sums."""
import numpy as np
import pytest

from candy_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("m", [2, 15, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("n,k", [(64, 64), (100, 250), (1000, 320), (2816, 384), (130, 448), (65, 2100)])
def test_narrow_tiles(dev, m, n, k):
    rng = np.random.default_rng(m + n * k)
    w = hip.bf16_bits(rng.standard_normal((n, k)))
    x = hip.bf16_values(hip.bf16_bits(rng.standard_normal((m, k))))
    wide, dense = hip.bf16_values(w).astype(np.float64), dev.dense(w)
    want = x.astype(np.float64) @ wide.T
    # f32 sums of exact products, in any order: K roundings of 2^-24 of the sum of magnitudes at most
    bound = (k + 1) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(wide).T)
    got, pos = dev.dense_matmul(dense, x, epilogue=hip.EPI_SQUARED_RELU), np.maximum(want, 0)
    assert np.all(np.abs(got - pos ** 2) <= (2 * pos + bound) * bound * 1.01 + 2.0 ** -8 * pos ** 2)
    # whole K in one order, whatever the tile: the f32 results of the other kernels, rounded
    plain = dev.dense_matmul(dense, x)
    assert np.array_equal(dev.dense_matmul(dense, x, epilogue=hip.EPI_ACT), hip.bf16_values(hip.bf16_bits(plain)))
