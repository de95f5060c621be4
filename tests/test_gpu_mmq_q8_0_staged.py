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


# Gate and up of a prompt with SiLU in the tiles (64 rows of each in turns of 32, so a producer's rows and slice lie elsewhere), two, three
# and five super-blocks, tiles of 256, 192 and 128 activation rows; against launches of their own on the tiles whose lanes load their
# own runs.  The other projections split K alike on either side.
@pytest.mark.gpu
@pytest.mark.parametrize("n,d_model,d_ffn", [(500, 768, 6144), (300, 512, 6144), (300, 768, 6144), (300, 1280, 6144), (257, 768, 9472)])
def test_gate_and_up_same_bits_as_loads_of_single_lanes(dev, n, d_model, d_ffn):
    c = dict(n_layers=1, d_model=d_model, n_heads=2, n_kv_heads=2, head_dim=128, d_ffn=d_ffn, vocab=256, max_pos=n, rms_eps=1e-5, rope_base=10000.0)
    m, fmt = hip.Llama(dev, **c), synth.Q8_0
    shapes = {hip.W_Q: (256, d_model), hip.W_K: (256, d_model), hip.W_V: (256, d_model), hip.W_O: (d_model, 256), hip.W_GATE: (d_ffn, d_model),
              hip.W_UP: (d_ffn, d_model), hip.W_DOWN: (d_model, d_ffn), hip.W_HEAD: (256, d_model), hip.W_EMBED: (256, d_model)}
    for kind, (rows, cols) in shapes.items():
        w = synth.random_weight(fmt, rows, cols, seed=kind, scale=synth.unit_scale(fmt))
        m.set_qweight(kind, -1 if kind in (hip.W_HEAD, hip.W_EMBED) else 0, dev.qtensor(fmt, rows, cols, w))
    for kind, layer in ((hip.W_ATTN_NORM, 0), (hip.W_FFN_NORM, 0), (hip.W_OUT_NORM, -1)):
        m.set_norm(kind, layer, np.ones(d_model, np.float32))
    tokens = [int(t) for t in np.random.default_rng(n).integers(0, 256, n)]

    def rows():
        m.prefill(tokens, 0, want_logits=False)
        return np.array(m.prompt_hidden(n))

    got = rows()
    dev.set_option("prefill.fold_silu", 0)
    dev.set_option("mmq.f16_shape", 3)
    try:
        want = rows()
    finally:
        dev.set_option("prefill.fold_silu", 1)
        dev.set_option("mmq.f16_shape", 0)
    assert np.isfinite(got).all() and np.array_equal(got.view(np.uint32), want.view(np.uint32))
