"""silu(gate) where the reciprocal of 1 + exp(-gate) is no normal number, times an infinite up: the prompt's tiles leave what the
launch of its own leaves, -infinity and not 0 times infinity."""
import numpy as np
import pytest

from candy_amd import hip, synth

D, FFN, N = 256, 6144, 300


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def q8_rows(scale, level, rows, cols=D):
    """One value per row, in column 0: level times the row's scale; zeros behind it."""
    b = np.zeros((rows, cols // 32, 34), np.uint8)
    b[:, 0, :2] = np.broadcast_to(np.asarray(scale, np.float16), (rows,))[:, None].view(np.uint8)
    b[:, 0, 2] = np.broadcast_to(np.asarray(level, np.int8), (rows,)).view(np.uint8)
    return b.reshape(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("at", [-87.0, -87.6, -88.2, -89.5])
def test_far_below_zero_times_infinity(dev, at):
    m = hip.Llama(dev, n_layers=1, d_model=D, n_heads=2, n_kv_heads=2, head_dim=128, d_ffn=FFN, vocab=256, max_pos=N, rms_eps=1e-5,
                  rope_base=10000.0)
    put = lambda kind, layer, blocks, rows, cols=D: m.set_qweight(kind, layer, dev.qtensor(synth.Q8_0, rows, cols, blocks))
    for kind in (hip.W_Q, hip.W_K, hip.W_V, hip.W_O):
        put(kind, 0, q8_rows(0, 0, D), D)  # the residual stream stays the embedding's: ones, which the norm leaves
    ones = np.zeros((256, D // 32, 34), np.uint8)
    ones[:, :, :2] = np.full((256, D // 32, 1), 1 / 64, np.float16).view(np.uint8)
    ones[:, :, 2:] = 64
    put(hip.W_EMBED, -1, ones.reshape(-1), 256)
    put(hip.W_GATE, 0, q8_rows(at / 127, 127, FFN), FFN)  # every gate value within 0.05 of `at`
    # up: 1, and in the row of every 64th value a weight that fp16 does not hold
    scale, level = np.full(FFN, 1 / 64), np.full(FFN, 64)
    scale[::64], level[::64] = 1000, 127
    put(hip.W_UP, 0, q8_rows(scale, level, FFN), FFN)
    put(hip.W_DOWN, 0, synth.random_weight(synth.Q8_0, D, FFN, seed=1, scale=synth.unit_scale(synth.Q8_0)), D, FFN)
    put(hip.W_HEAD, -1, synth.random_weight(synth.Q8_0, 256, D, seed=2, scale=synth.unit_scale(synth.Q8_0)), 256)
    for kind, layer in ((hip.W_ATTN_NORM, 0), (hip.W_FFN_NORM, 0), (hip.W_OUT_NORM, -1)):
        m.set_norm(kind, layer, np.ones(D, np.float32))

    def hidden():
        m.prefill(list(range(256)) + list(range(N - 256)), 0, want_logits=False)
        return m.prompt_hidden(N)

    got = hidden()
    dev.set_option("prefill.fold_silu", 0)
    try:
        want = hidden()
    finally:
        dev.set_option("prefill.fold_silu", 1)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.isnan(want).all() == (at > -88.7)  # from -88.73 exp overflows: silu is -0 there, and 0 times infinity no number
    assert np.array_equal(got[~np.isnan(got)].view(np.uint32), want[~np.isnan(want)].view(np.uint32))
