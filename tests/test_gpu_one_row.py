"""The one-row kernels of the bfloat16 decoders at the edges of their steps: K one step, two, a value past either, past the piece of the
row that LDS holds; one, two and four weight rows a wavefront; experts whose inner widths end anywhere in the last step."""
import numpy as np
import pytest

from candy_amd import hip
from oracle import suvazen_ref as ref
from tests import suvazen_models as sm
from tests.test_gpu_gulisun import Experts, own
from tests.test_gpu_suvazen import build, rel

pytestmark = pytest.mark.gpu
ACTS = [pytest.param(hip.ACT_F32, id="f32"), pytest.param(hip.ACT_BF16, id="bf16")]


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("rows,cols", [(200, 2048), (200, 2049), (130, 4096), (130, 4160), (70, 8192), (70, 8256), (70, 12300), (40, 16384),
                                       (40, 16390), (40, 33000), (8192, 1024), (8190, 2049), (8192, 4096), (17000, 1030), (16500, 3100)])
def test_contraction_of_one_row(dev, rows, cols, act):
    rng = np.random.default_rng(rows + cols)
    w = sm.to_bf16(rng.standard_normal((rows, cols)) * cols ** -0.5)
    dw = dev.dense(sm.bits_of(w))
    x = rng.standard_normal((1, cols)).astype(np.float32)
    xa = sm.to_bf16(x) if act == hip.ACT_BF16 else x
    want = xa.astype(np.float64) @ w.T.astype(np.float64)
    assert rel(dev.dense_matmul(dw, x, act), want) < 3e-6 + 3e-8 * cols ** 0.5  # f32 sums of `cols` terms
    dw.free()


@pytest.mark.parametrize("width,ff", [(2048, 8192), (2050, 300), (4096, 2600), (4200, 100), (6400, 64), (8300, 16400)])
def test_norms_in_the_prologue(dev, width, ff):
    """A token fed alone (norms in front of the contraction) against the oracle and against the same token as a prompt's."""
    cfg = sm.config([(sm.mixer(4, 2, 32, 64, 32, 10000.0, None, 0.18, 20.0), ff)] * 2, width, 96)
    w = sm.weights(cfg, seed=width)
    tokens = [int(t) for t in np.random.default_rng(1).integers(0, 96, 5)]
    want = ref.forward(cfg, w, tokens)
    m = build(dev, cfg, w, hip.ACT_BF16)
    alone = np.concatenate([m.feed([t], i, [0]) for i, t in enumerate(tokens)])
    assert rel(alone, want) < 4e-2   # bfloat16 activations
    steps = np.stack([m.decode(t, i)[1] for i, t in enumerate(tokens)])
    assert rel(steps, want) < 4e-2
    m.free()


@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("d,experts,top,ff,shared", [(2048, 6, 3, 640, 2176), (2112, 6, 3, 640, 128), (300, 4, 2, 2048, None), (300, 9, 3, 1400, 60),
                                                     (4200, 3, 1, 64, 512), (128, 80, 5, 1000, 3200)])
def test_experts_of_one_row(dev, d, experts, top, ff, shared, act):
    case = Experts(dev, d, experts, top, ff, shared, d)
    x = sm.to_bf16(np.random.default_rng(d).standard_normal((3, d)) * 1.2)
    want = case.oracle(x)[0]
    rows = np.concatenate([dev.experts(case.spec, act, case.dense, x[t:t + 1], decode=True) for t in range(3)])
    assert own(rows, want) < (1e-5 if act == hip.ACT_F32 else 1.5e-2)


# rows that leave LDS no more than the scores and the choice, which the zeros share where they are in it
@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("d,experts,top", [(16320, 40, 12), (16320, 2, 1), (16256, 100, 14)])
def test_experts_of_the_widest_rows(dev, d, experts, top, act):
    case = Experts(dev, d, experts, top, 5, 70, top)
    x = sm.to_bf16(np.random.default_rng(d).standard_normal((1, d)) * 1.2)
    rows = dev.experts(case.spec, act, case.dense, x, decode=True)
    assert own(rows, case.oracle(x)[0]) < (1e-5 if act == hip.ACT_F32 else 1.5e-2)


# wavefronts wholly behind the last row, which is a chosen expert's: workgroups of 11 x 1, 9 x 4 and 11 x 4 rows on 256 CUs
@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("d,experts,top,ff", [(200, 4, 2, 1344), (136, 7, 6, 1408), (136, 64, 8, 1408)])
def test_experts_without_a_shared_one_and_wavefronts_without_rows(dev, d, experts, top, ff, act):
    case = Experts(dev, d, experts, top, ff, None, d)
    x = sm.to_bf16(np.random.default_rng(d).standard_normal((3, d)) * 1.2)
    want = case.oracle(x)[0]
    rows = np.concatenate([dev.experts(case.spec, act, case.dense, x[t:t + 1], decode=True) for t in range(3)])
    assert own(rows, want) < (1e-5 if act == hip.ACT_F32 else 1.5e-2)
