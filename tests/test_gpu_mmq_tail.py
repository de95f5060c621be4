"""Grids of fp16 tiles whose last round is split along K: against the oracle, and against tiles that are all whole."""
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


def whole(dev, call):
    dev.set_option("mmq.f16_split", 1)
    try:
        return call()
    finally:
        dev.set_option("mmq.f16_split", 0)


# one tile behind a round (rows that end inside it, and not at a multiple of four; one activation row in it), two (192 and 256
# activation rows wide), half a round (two splits of unequal length; Q4_K: whole), a third, K of eight and nine super-blocks, two full
# rounds (Q4_K: none)
@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML])
@pytest.mark.parametrize("rows,cols,m", [(10985, 2048, 513), (32770, 2048, 200), (11008, 2304, 577), (11008, 2048, 700), (16384, 2304, 520),
                                         (14336, 2048, 560), (11008, 2048, 1400)])
def test_last_round_in_splits(dev, fmt, rows, cols, m):
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    got = dev.qmatmul(q, x)
    want = whole(dev, lambda: dev.qmatmul(q, x))
    # the same products in sums of another order: a few 2^-24 of sums of 2048 values and more
    assert np.max(np.abs(got - want)) <= 2e-6 * np.max(np.abs(want))
    sub, some = np.unique(np.r_[0:rows:499, rows - 130:rows]), np.unique(np.r_[0, 191, 192, 255, 256, 511, 512, m - 1])
    some = some[some < m]
    part = np.ascontiguousarray(w.reshape(rows, -1)[sub]).reshape(-1)
    want = o.qmatmul(fmt, part, len(sub), cols, x[some])
    # weight and activation of a product are each rounded to fp16, by up to 2^-11 of it and evenly within that: sqrt(2 / 3) 2^-11 of the
    # root of the products' sum of squares; six times that for the largest of some thousand
    values = o.dequantize(fmt, part).reshape(len(sub), cols).astype(np.float64)
    spread = np.sqrt((x[some].astype(np.float64) ** 2) @ (values ** 2).T) * (2 / 3) ** 0.5 * 2.0 ** -11
    assert np.all(np.abs(got[some][:, sub] - want) <= 6 * spread)


def test_three_tensors_and_a_residual(dev):
    """A prompt whose q / k / v (one grid, tiles of the last round in two of the tensors) and o (with the residual) end in splits."""
    n, d = 2100, 4096
    c = dict(n_layers=1, d_model=d, n_heads=32, n_kv_heads=32, head_dim=128, d_ffn=256, vocab=256, max_pos=n, rms_eps=1e-5, rope_base=10000.0)
    m, rng, fmt = hip.Llama(dev, **c), np.random.default_rng(3), synth.Q4_K
    shapes = {hip.W_Q: (d, d), hip.W_K: (d, d), hip.W_V: (d, d), hip.W_O: (d, d), hip.W_GATE: (256, d), hip.W_UP: (256, d), hip.W_DOWN: (d, 256)}
    for s, (at, (rows, cols)) in enumerate(shapes.items()):
        m.set_qweight(at, 0, dev.qtensor(fmt, rows, cols, synth.random_weight(fmt, rows, cols, seed=s, scale=synth.unit_scale(fmt))))
    for at, layer in ((hip.W_ATTN_NORM, 0), (hip.W_FFN_NORM, 0), (hip.W_OUT_NORM, -1)):
        m.set_norm(at, layer, (1 + 0.1 * rng.standard_normal(d)).astype(np.float32))
    for s, at in enumerate((hip.W_HEAD, hip.W_EMBED)):
        m.set_qweight(at, -1, dev.qtensor(fmt, 256, d, synth.random_weight(fmt, 256, d, seed=20 + s, scale=synth.unit_scale(fmt))))
    tokens = [int(t) for t in rng.integers(0, 256, n)]
    got = np.array(m.prefill(tokens, 0)[1])
    want = whole(dev, lambda: np.array(m.prefill(tokens, 0)[1]))
    # levels of the quantized activations that lie at a half may go the other way: 1 / 254 of a block's largest value each
    assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
