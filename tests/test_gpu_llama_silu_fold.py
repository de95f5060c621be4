"""Prompts whose gate / up launch leaves silu(gate) * up as the fp16 image of its quantization: the same bits as the launches of
their own, at the tiles' edges and where the products overflow."""
import numpy as np
import pytest

from candy_amd import hip, synth

KINDS = {"q": hip.W_Q, "k": hip.W_K, "v": hip.W_V, "o": hip.W_O, "gate": hip.W_GATE, "up": hip.W_UP, "down": hip.W_DOWN}


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def model(dev, fmt, d_ffn, gain, max_pos):
    c = dict(n_layers=1, d_model=256, n_heads=2, n_kv_heads=2, head_dim=128, d_ffn=d_ffn, vocab=256, max_pos=max_pos, rms_eps=1e-5,
             rope_base=10000.0)
    m, rng = hip.Llama(dev, **c), np.random.default_rng(d_ffn)
    for s, (kind, at) in enumerate(KINDS.items()):
        rows, cols = (d_ffn, 256) if kind in ("gate", "up") else (256, d_ffn) if kind == "down" else (256, 256)
        m.set_qweight(at, 0, dev.qtensor(fmt, rows, cols, synth.random_weight(fmt, rows, cols, seed=s, scale=synth.unit_scale(fmt))))
    for at, layer, by in ((hip.W_ATTN_NORM, 0, 1), (hip.W_FFN_NORM, 0, gain), (hip.W_OUT_NORM, -1, 1)):
        m.set_norm(at, layer, (by * (1 + 0.1 * rng.standard_normal(256))).astype(np.float32))
    for s, at in enumerate((hip.W_HEAD, hip.W_EMBED)):
        m.set_qweight(at, -1, dev.qtensor(fmt, 256, 256, synth.random_weight(fmt, 256, 256, seed=20 + s, scale=synth.unit_scale(fmt))))
    return m


# 128 x 256 tiles (whole, and a ragged second column); 128 x 192 (one row past 256, and 300); 128 x 128 where they need no more
# rounds (three, five columns of tiles, the last of 1 and 128 rows); products that fp16 scales, and f32, cannot hold
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML])
@pytest.mark.parametrize("n,d_ffn,gain", [(256, 12288, 1), (257, 6144, 1), (500, 6400, 0.01), (257, 9472, 1), (640, 5632, 1), (300, 6144, 30),
                                          (300, 6144, 1e20)])
def test_folded_silu_gives_the_bits_of_its_own_launch(dev, fmt, n, d_ffn, gain):
    m = model(dev, fmt, d_ffn, gain, n)
    tokens = [int(t) for t in np.random.default_rng(n).integers(0, 256, n)]
    got = np.array(m.prefill(tokens, 0)[1])
    dev.set_option("prefill.fold_silu", 0)
    try:
        want = np.array(m.prefill(tokens, 0)[1])
    finally:
        dev.set_option("prefill.fold_silu", 1)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~np.isnan(got)].view(np.uint32), want[~np.isnan(want)].view(np.uint32))
    assert gain > 1 or not np.isnan(got).any()
