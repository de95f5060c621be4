"""The large tiles of bfloat16 contractions at their edges: rows of the last tile (quarters of 32 and 64 rows), weight rows
past the last tile, one stage of K and odd numbers of stages, every epilogue, rows dealt to experts."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip
from oracle import gulisun_ref as ref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def bf16(x):
    return hip.bf16_values(hip.bf16_bits(x))


# The tile goes by the shape: 128 activation rows up to a few hundred, 256 beyond; 128 .. 256 weight rows.
@pytest.mark.parametrize("m", [65, 97, 128, 129, 200, 256, 257, 321, 512, 800])
@pytest.mark.parametrize("n,k", [(64, 64), (200, 100), (1000, 192), (2600, 320), (5100, 448), (14300, 128)])
def test_tiles(dev, m, n, k):
    rng = np.random.default_rng(m * n + k)
    w = hip.bf16_bits(rng.standard_normal((n, k)))
    x = bf16(rng.standard_normal((m, k)))
    wide = hip.bf16_values(w).astype(np.float64)
    want = x.astype(np.float64) @ wide.T
    # f32 sums of exact products, in any order: K roundings of 2^-24 of the sum of magnitudes at most
    bound = (k + 1) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(wide).T)
    dense = dev.dense(w)
    assert np.all(np.abs(dev.dense_matmul(dense, x) - want) <= bound)
    # rounded to bfloat16 (half of 2^-8) behind the epilogue, which doubles a relative error
    got = dev.dense_matmul(dense, x, epilogue=hip.EPI_ACT)
    assert np.all(np.abs(got - want) <= bound + 2.0 ** -8 * np.abs(want))
    got, pos = dev.dense_matmul(dense, x, epilogue=hip.EPI_SQUARED_RELU), np.maximum(want, 0)
    assert np.all(np.abs(got - pos ** 2) <= (2 * pos + bound) * bound * 1.01 + 2.0 ** -8 * pos ** 2)
    got = dev.dense_matmul(dense, x, epilogue=hip.EPI_SOFTCAP, scale=0.5, cap=20.0)
    assert np.all(np.abs(got - 20 * np.tanh(want / 40)) <= bound + 1e-5)


def dealt(dev, tokens, skew, d, experts, top, ff):
    rng = np.random.default_rng(tokens)
    router = bf16(rng.standard_normal((experts, d)) * 0.3)
    router[0] += np.float32(skew * 0.0625)
    up, down = (bf16(rng.standard_normal((experts, *s)) * 0.1) for s in ((ff, d), (d, ff)))
    x = bf16(rng.standard_normal((tokens, d)) + 0.5)
    w = {"p.router": bf16(router).astype(np.float64)}
    for e in range(experts):
        w[f"p.e{e}.up"], w[f"p.e{e}.down"] = up[e].astype(np.float64), down[e].astype(np.float64)
    want = ref.experts(x.astype(np.float64), w, "p", {"router": {"experts": experts, "top": top}})
    padded = np.zeros((experts, -(-ff // 64) * 64, d), np.float32)
    padded[:, :ff] = up
    weights = {"router": dev.dense(hip.bf16_bits(router)), "up": dev.dense(hip.bf16_bits(padded.reshape(-1, d))),
               "down": dev.dense(hip.bf16_bits(down.reshape(-1, ff)))}
    spec = hip.ExpertSpec(n_experts=experts, top=top, d_ff=ff, shared_ff=0)
    got, ids, _ = dev.experts(spec, hip.ACT_BF16, weights, x)
    assert np.array_equal(ids, ref.route(x.astype(np.float64), w["p.router"], top)[0])
    # the inner activations are rounded to bfloat16 once: 2^-9 of each, of random sign
    assert np.max(np.abs(got - want)) <= 2.0 ** -7 * np.max(np.abs(want))
    assert np.sqrt(np.mean((got - want) ** 2)) <= 2.0 ** -8 * np.sqrt(np.mean(want ** 2))


@pytest.mark.parametrize("tokens,skew", [(150, 0.0), (300, 0.0), (300, 3.0), (700, 1.0)])
def test_rows_dealt_to_experts(dev, tokens, skew):
    dealt(dev, tokens, skew, 192, 3, 2, 300)


# Contractions long enough for the large tiles: 128 weight rows each while all tiles are on the chip at once, 256 (up) beyond
@pytest.mark.parametrize("tokens,skew,experts,ff", [(300, 0.0, 3, 800), (300, 3.0, 3, 800), (700, 1.0, 3, 1100), (1600, 0.0, 20, 830), (1700, 1.0, 20, 1100)])
def test_rows_dealt_to_experts_large_tiles(dev, tokens, skew, experts, ff):
    lib, padded = hip.lib(), -(-ff // 64) * 64
    assert lib.candy_test_grouped_tile_rows(experts, ctypes.c_int64(2 * tokens), ctypes.c_int64(padded)) == 128
    assert lib.candy_test_grouped_weight_rows(256, experts, ctypes.c_int64(2 * tokens), padded) == (256 if experts == 20 else 128)
    dealt(dev, tokens, skew, 192, experts, 2, ff)
