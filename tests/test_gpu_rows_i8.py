"""The exact contraction of 3 to 255 activation rows with K dealt to wavefronts: every tile shape and its edges, against the
oracle, the int8 tile and vector kernels (other order of f32 sums) and between the entry points."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o

FORMATS = [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML]
# Weight rows (off the strips of 16 and off the float4 stores), values per row (one super-block; fewer than, as many as and one
# more than the wavefronts), activation rows on both sides of every tile's edge; one, two and four strips per workgroup.
SHAPES = [(4099, 256, m) for m in (5, 16, 33, 64)] + [(1030, 1024, m) for m in (5, 17, 48, 49, 255)] + \
         [(258, 4352, m) for m in (16, 17, 65)] + [(2052, 2304, m) for m in (17, 32, 48, 64, 130)] + \
         [(4096, 4096, 18), (16500, 256, 7), (12500, 256, 31), (16500, 256, 40), (16500, 256, 50), (5000, 1024, 3)] + \
         [(4100, 256, 17), (11000, 256, 32), (8200, 1024, 25), (1500, 1024, 80), (3080, 512, 192), (1030, 2304, 129), (8200, 512, 255)]


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    d.set_option("rows.i8", 2)  # whatever the dispatch would take
    yield d
    d.close()


def rel_err(got, want):
    return float(np.max(np.abs(got.astype(np.float64) - want)) / np.max(np.abs(want)))


def exact(dev, w, x):
    """candy_hip_qmatmul_qact: the exact kernels up to 255 rows."""
    L, act = hip.lib(), ctypes.c_void_p()
    m, cols = x.shape
    src, dst = dev.alloc(x.nbytes), dev.alloc(4 * m * w.rows)
    src.upload(x)
    hip._check(L.candy_hip_qact_create(dev.handle, m, cols, ctypes.byref(act)))
    hip._check(L.candy_hip_qact_quantize(act, src.ptr, m, cols))
    hip._check(L.candy_hip_qmatmul_qact(dev.handle, w.handle, act, dst.ptr))
    out = dst.download(np.float32, m * w.rows).reshape(m, w.rows)
    hip._check(L.candy_hip_qact_free(act))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,cols,m", SHAPES)
def test_rows_against_oracle_and_other_kernels(dev, fmt, rows, cols, m):
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    got = exact(dev, q, x)
    assert np.array_equal(got.view(np.uint32), exact(dev, q, x).view(np.uint32))
    dev.set_option("rows.i8", 0)
    try:
        other = exact(dev, q, x)
    finally:
        dev.set_option("rows.i8", 2)
    # exact integer dots of 32 values; K / 32 products of two scales and their sum in f32, in two orders
    assert rel_err(got, other) <= 2e-6
    sub = np.arange(m) if m <= 16 else np.unique(np.r_[0, 15, 16, m // 2, m - 1])
    want = o.qmatmul(fmt, w, rows, cols, x[sub])
    assert rel_err(got[sub], want) <= 2e-5
    if m <= 16:  # f32 rows and Q8_0 blocks go through other kernels into the same operands
        assert np.array_equal(dev.qmatmul(q, x).view(np.uint32), dev.qmatmul_q8(q, dev.quantize_q8_0(x), m).view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
def test_a_row_reaches_its_own_results_only(dev, fmt):
    # The image of 5 rows is a tile of 16, and planar quants fill their own rows of it only.  What the call before left in rows 5 to
    # 14 of the same tile, here scales that are infinite and sums that are no numbers, must not be seen.
    w = synth.random_weight(fmt, 4099, 512, seed=3)
    q = dev.qtensor(fmt, 4099, 512, w)
    x = synth.random_activations(15, 512, seed=4)
    want = exact(dev, q, x[:5])
    x[5:] = np.inf
    assert not np.isfinite(exact(dev, q, x)[5:]).any()
    assert np.array_equal(exact(dev, q, x[:5]).view(np.uint32), want.view(np.uint32))
    assert np.all(np.isfinite(want)) and np.array_equal(dev.qmatmul(q, x[:5]).view(np.uint32), want.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q6_K, synth.Q8_0])
def test_a_prompt_sees_its_own_rows_only(dev, fmt):
    # The same for the operands that a prompt's launches write: 15 tokens, ten of them of an infinite embedding, then five
    c = dict(n_layers=1, d_model=512, n_heads=4, n_kv_heads=2, head_dim=128, d_ffn=1024, vocab=256, max_pos=32, rms_eps=1e-5, rope_base=10000.0)
    shapes = {hip.W_Q: (512, 512), hip.W_K: (256, 512), hip.W_V: (256, 512), hip.W_O: (512, 512), hip.W_GATE: (1024, 512), hip.W_UP: (1024, 512),
              hip.W_DOWN: (512, 1024)}
    embed = synth.random_weight(synth.Q8_0, 256, 512, seed=9, scale=synth.unit_scale(synth.Q8_0))
    embed.reshape(256, 16, 34)[255, :, :2] = np.full((16, 1), np.inf, np.float16).view(np.uint8)

    def model():
        m = hip.Llama(dev, **c)
        for kind, (r, k) in shapes.items():
            m.set_qweight(kind, 0, dev.qtensor(fmt, r, k, synth.random_weight(fmt, r, k, seed=kind, scale=synth.unit_scale(fmt))))
        for kind, layer in ((hip.W_ATTN_NORM, 0), (hip.W_FFN_NORM, 0), (hip.W_OUT_NORM, -1)):
            m.set_norm(kind, layer, np.ones(512, np.float32))
        m.set_qweight(hip.W_EMBED, -1, dev.qtensor(synth.Q8_0, 256, 512, embed))
        m.set_qweight(hip.W_HEAD, -1, dev.qtensor(synth.Q8_0, 256, 512, embed))
        return m

    def hidden(m, tokens):
        m.prefill(tokens, 0, want_logits=False)
        return m.prompt_hidden(len(tokens))

    tokens = [3, 1, 4, 1, 5]
    want, m = hidden(model(), tokens), model()
    assert np.isfinite(want).all() and not np.isfinite(hidden(m, tokens + [255] * 10)[5:]).any()
    assert np.array_equal(hidden(m, tokens).view(np.uint32), want.view(np.uint32))


# Up to eight rows share the columns of a product in two groups: as many strips per workgroup and wavefronts as there are, the last
# column and the first row count past it, against the same rows in a batch of 16 columns.
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,cols", [(16, 256), (1030, 4352), (4099, 512), (8200, 256), (16500, 768)])
def test_two_groups_of_columns(dev, fmt, rows, cols):
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    x = synth.random_activations(16, cols, seed=cols)
    q = dev.qtensor(fmt, rows, cols, w)
    whole = exact(dev, q, x)
    for m in (3, 7, 8, 9):
        assert rel_err(exact(dev, q, x[:m]), whole[:m]) <= 2e-6  # two orders of f32 sums, as above
