"""Prompt attention in bfloat16 at the edges of its tiles: window attention with rows of 64 and 128 values, whose tiles go to
LDS by direct loads, and latent attention with keys and values of whole 64s."""
import numpy as np
import pytest

from candy_amd import hip
from tests import gulisun_models as gm
from tests import suvazen_models as sm
from tests.test_gpu_gulisun import Latent
from tests.test_gpu_suvazen import device_attention, oracle_attention, rel

pytestmark = pytest.mark.gpu

# what is left against the oracle, which rounds the stored operands like the device: results in bfloat16 (2^-9 of each) and
# operands that round the other way (2^-8 of a few), summed over a row: 1.2e-2, and 1.5e-2 where the oracle leaves the
# rebuilt keys and values unrounded
WINDOW_TOL, LATENT_TOL = 1.2e-2, 1.5e-2


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


# heads, kv heads, dim, window, scale, cap: heads that deal evenly to the XCDs and not; widths that fill their rows and not;
# windows within a tile, at a tile's edge and none; a scale of either sign and of 0 (all keys alike)
WINDOW = [(8, 2, 64, None, 0.15, None), (8, 8, 128, 33, 0.09, 20.0), (3, 1, 50, 64, -0.2, None), (6, 2, 118, 31, -0.1, 30.0),
          (16, 2, 128, 65, 0.0, None), (5, 5, 64, 1, 0.3, 5.0)]


@pytest.mark.parametrize("heads,kv_heads,dim,window,scale,cap", WINDOW)
def test_window(dev, heads, kv_heads, dim, window, scale, cap):
    n = 195
    mx = sm.mixer(heads, kv_heads, dim, window, 2 * (dim // 4), 1000.0, None, scale, cap)
    rng = np.random.default_rng(dim)
    q = (rng.standard_normal((n, heads, dim)) * 1.5).astype(np.float32)
    k = (rng.standard_normal((n, kv_heads, dim)) * 1.5).astype(np.float32)
    sink = rng.standard_normal(heads).astype(np.float32)
    for s in (sink, None):
        want = oracle_attention(mx, q.astype(np.float64), k.astype(np.float64), s, hip.ACT_BF16)
        for portions in ([n], [31, 2, 32, 63, 67], [65, 64, 33, 33]):
            assert rel(device_attention(dev, mx, q, k, s, hip.ACT_BF16, portions), want) < WINDOW_TOL, (s is None, portions)


# sinks of -infinity and of the type's lowest value (exp(sink) = 0: heads without one) where a query's first tile of 32 keys is
# wholly in front of its window, the window within a tile, at its edge and longer
@pytest.mark.parametrize("dim,window", [(64, 32), (128, 32), (64, 64), (128, 50), (64, 1)])
def test_window_sink_of_no_weight(dev, dim, window):
    n, heads = 195, 8
    rng = np.random.default_rng(window)
    q = (rng.standard_normal((n, heads, dim)) * 1.5).astype(np.float32)
    k = (rng.standard_normal((n, 2, dim)) * 1.5).astype(np.float32)
    sink = np.array([-np.inf, 0.5, -np.inf, -3.4e38, -1e30, -np.inf, -2.0, -3.4e38], np.float32)
    for cap in (None, 20.0):
        mx = sm.mixer(heads, 2, dim, window, 2 * (dim // 4), 1000.0, None, 0.1, cap)
        want = oracle_attention(mx, q.astype(np.float64), k.astype(np.float64), sink, hip.ACT_BF16)
        assert np.all(np.isfinite(want))
        for portions in ([n], [31, 2, 32, 63, 67]):
            assert rel(device_attention(dev, mx, q, k, sink, hip.ACT_BF16, portions), want) < WINDOW_TOL, (cap, portions)


# heads, dim, rotated, values: keys and values of whole 64s (rotated parts of 32 and more, also ragged ones)
LATENT = [(8, 32, 32, 64), (3, 64, 64, 64), (2, 96, 18, 50), (16, 64, 40, 128), (5, 128, 64, 64), (8, 128, 64, 128), (1, 32, 150, 100),
          (4, 192, 64, 128), (2, 32, 224, 128), (2, 256, 0, 128)]


@pytest.mark.parametrize("heads,dim,rot,vdim", LATENT)
def test_latent(dev, heads, dim, rot, vdim):
    n = 195
    for scale, seed in ((None, 1), (-0.5 * (dim + rot) ** -0.5, 2)):
        case = Latent(dev, gm.latent(heads, dim, rot, vdim, 96, 40, 500.0, abs(scale) if scale else None)["mixer"], n, seed)
        if scale:  # (the inputs are drawn for its size)
            case.m["scale"] = scale
            case.spec.scale = scale
        sink = np.random.default_rng(seed).standard_normal(heads).astype(np.float32)
        for s in (sink, None):
            want = case.oracle(s, hip.ACT_BF16)
            for portions in ([n], [31, 2, 32, 63, 67], [65, 64, 33, 33]):
                assert rel(case.device(s, hip.ACT_BF16, portions), want) < LATENT_TOL, (scale, s is None, portions)
