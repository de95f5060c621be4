"""Prompt attention on the matrix cores against the vector-ALU kernel, at the edges of its tiles: one-layer models whose
feed-forward is switched off (zero weights), so that the hidden rows are x + Wo . q8(attention)."""
import numpy as np
import pytest

from candy_amd import hip, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def one_layer(dev, heads, kv_heads, head_dim, max_pos):
    d = heads * head_dim
    cfg = dict(n_layers=1, d_model=d, n_heads=heads, n_kv_heads=kv_heads, head_dim=head_dim, d_ffn=256, vocab=256, max_pos=max_pos,
               rms_eps=1e-5, rope_base=10000.0)
    model, kd, f = hip.Llama(dev, **cfg), kv_heads * head_dim, synth.Q8_0
    scale = synth.unit_scale(f)
    for i, (kind, rows, cols) in enumerate(((hip.W_Q, d, d), (hip.W_K, kd, d), (hip.W_V, kd, d), (hip.W_O, d, d), (hip.W_GATE, 256, d),
                                            (hip.W_UP, 256, d), (hip.W_HEAD, 256, d), (hip.W_EMBED, 256, d))):
        layer = -1 if kind in (hip.W_HEAD, hip.W_EMBED) else 0
        # q and k wide enough that the weights of a row differ by orders of magnitude
        model.set_qweight(kind, layer, dev.qtensor(f, rows, cols, synth.random_weight(f, rows, cols, 50 + i, scale * (2 if i < 2 else 1))))
    model.set_qweight(hip.W_DOWN, 0, dev.qtensor(f, d, 256, np.zeros(synth.weight_nbytes(f, d, 256), np.uint8)))
    for kind, layer in ((hip.W_ATTN_NORM, 0), (hip.W_FFN_NORM, 0), (hip.W_OUT_NORM, -1)):
        model.set_norm(kind, layer, np.ones(d, np.float32))
    return model


# (heads, kv heads, head_dim): shared kv heads; heads that do not divide over the XCDs; no sharing; and a head count with
# which a long prompt takes the 128-query form
SHAPES = [(8, 2, 64), (6, 2, 128), (4, 4, 64), (32, 4, 64), (8, 8, 128)]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("heads,kv_heads,head_dim", SHAPES)
def test_tiles_edges_against_the_vector_kernel(dev, heads, kv_heads, head_dim, f16):
    lengths = [(1, 0), (31, 1), (32, 0), (33, 0), (64, 0), (65, 63), (130, 64), (300, 97)] + ([(1100, 1061)] if heads == 32 else [])
    model = one_layer(dev, heads, kv_heads, head_dim, 1104)
    if f16:
        model.set_kv_f16(True)
    rng = np.random.default_rng(heads * head_dim)
    for n, cut in lengths:  # the whole prompt, and (cut > 0) the same in two passes
        tokens = [int(t) for t in rng.integers(0, 256, n)]
        got = {}
        try:
            for valu in (1, 0):
                dev.set_option("prefill.attention_valu", valu)
                model.prefill(tokens, 0, want_logits=False)
                got[valu] = model.prompt_hidden(n)
                if cut and not valu:
                    model.prefill(tokens[:cut], 0, want_logits=False)
                    model.prefill(tokens[cut:], cut, want_logits=False)
                    got["cut"] = model.prompt_hidden(n - cut)
        finally:
            dev.set_option("prefill.attention_valu", 0)
        # The two kernels agree to about 1e-6; a level of the quantizer behind them that falls the other way for it is
        # 1/127 of its block's range in one of K = heads * head_dim products of random sign: 1/127/sqrt(K) of the largest
        # result per level, and a few of a row's levels may move.
        bar = 8 / 127 / np.sqrt(heads * head_dim)
        top = np.max(np.abs(got[1]))
        assert np.max(np.abs(got[0] - got[1])) <= bar * top, (n, "whole")
        assert np.mean(np.abs(got[0] - got[1])) <= 1e-4 * top, (n, "whole, mean")
        if cut:
            # (below 256 rows and above it the projections round differently: fp16 operands, 3e-4 per contraction)
            mixed = n >= 256
            assert np.max(np.abs(got["cut"] - got[1][cut:])) <= (bar + 4e-3 if mixed else bar) * top, (n, cut)


# ------------------------------------------------------------------ accuracy
def mirror(dev, heads, kv_heads, head_dim, max_pos, q_std, k_std):
    """One layer whose hidden rows are (but for x, a thousandth of them) the quantized attention itself: Wo is the identity.  q and k
    are about q_std and k_std wide, v about 1."""
    d, kd, f = heads * head_dim, kv_heads * head_dim, synth.Q8_0
    model = hip.Llama(dev, n_layers=1, d_model=d, n_heads=heads, n_kv_heads=kv_heads, head_dim=head_dim, d_ffn=256, vocab=256, max_pos=max_pos,
                      rms_eps=1e-12, rope_base=10000.0)

    def matrix(rows, cols, seed, std):  # levels of +-127 / sqrt(3) rms
        rng = np.random.default_rng(seed)
        w = np.zeros((rows * cols // 32, 34), np.uint8)
        w[:, :2] = np.full((len(w), 1), std / (127 / 3 ** 0.5 * cols ** 0.5), np.float16).view(np.uint8)
        w[:, 2:] = rng.integers(-127, 128, (len(w), 32)).astype(np.int8).view(np.uint8)
        return dev.qtensor(f, rows, cols, w.reshape(-1))

    eye = np.zeros((d * d // 32, 34), np.uint8)
    eye[:, :2] = np.full((len(eye), 1), 1 / 127, np.float16).view(np.uint8)
    i = np.arange(d)
    eye[i * (d // 32) + i // 32, 2 + i % 32] = 127
    for kind, w in ((hip.W_Q, matrix(d, d, 1, q_std)), (hip.W_K, matrix(kd, d, 2, k_std)), (hip.W_V, matrix(kd, d, 3, 1.0)),
                    (hip.W_O, dev.qtensor(f, d, d, eye.reshape(-1))), (hip.W_GATE, matrix(256, d, 4, 1.0)), (hip.W_UP, matrix(256, d, 5, 1.0)),
                    (hip.W_DOWN, dev.qtensor(f, d, 256, np.zeros(synth.weight_nbytes(f, d, 256), np.uint8)))):
        model.set_qweight(kind, 0, w)
    model.set_qweight(hip.W_HEAD, -1, matrix(256, d, 6, 1.0))
    model.set_qweight(hip.W_EMBED, -1, matrix(256, d, 7, 1e-3 * d ** 0.5))
    for kind, layer in ((hip.W_ATTN_NORM, 0), (hip.W_FFN_NORM, 0), (hip.W_OUT_NORM, -1)):
        model.set_norm(kind, layer, np.ones(d, np.float32))
    return model


def both(dev, model, tokens, pos0=0):
    """Hidden rows by the vector-ALU kernel and by the matrix cores."""
    got = []
    try:
        for valu in (1, 0):
            dev.set_option("prefill.attention_valu", valu)
            model.prefill(tokens, pos0, want_logits=False)
            got.append(model.prompt_hidden(len(tokens)))
    finally:
        dev.set_option("prefill.attention_valu", 0)
    return got


# A level falls the other way where the two kernels' results, e of the block's largest value apart, lie on either side of its
# edge: a share of 2 * 127 * e.  f32 sums and exponentials that round at 2^-24 to 2^-22 leave e of 2^-21 at most: 1.2e-4, and 2e-4
# with room.  Weights of one 16-bit part (2^-12 each) are far past it.
SHARE = 2e-4
# (heads, kv heads, head_dim, f16 cache, q_std, k_std); queries past fp16's range, and keys near its end beside small queries:
# head_dim 64, whose parts stand for 32 bits
ACCURACY = [(8, 2, 64, False, 1.0, 1.0), (8, 2, 64, True, 1.0, 1.0), (6, 2, 128, False, 1.0, 1.0), (6, 2, 128, True, 1.0, 1.0),
            (32, 4, 64, False, 1.5, 1.5), (32, 4, 64, True, 1.5, 1.5), (8, 2, 64, True, 3e5, 1e-4), (8, 2, 64, False, 3e5, 1e-4),
            (8, 2, 64, True, 3e-4, 1e4), (8, 2, 64, False, 3e-4, 1e4)]


@pytest.mark.parametrize("heads,kv_heads,head_dim,f16,q_std,k_std", ACCURACY)
def test_levels_of_the_result(dev, heads, kv_heads, head_dim, f16, q_std, k_std):
    model = mirror(dev, heads, kv_heads, head_dim, 1104, q_std, k_std)
    if f16:
        model.set_kv_f16(True)
    rng = np.random.default_rng(head_dim)
    for n in (70, 300) + ((1100,) if heads == 32 else ()):
        want, got = both(dev, model, [int(t) for t in rng.integers(0, 256, n)])
        assert np.all(np.isfinite(want)) and np.all(np.isfinite(got)), n
        level = np.max(np.abs(want).reshape(n, -1, 32), axis=2, keepdims=True) / 127
        moved = np.abs(got - want).reshape(n, -1, 32) > 0.5 * level
        assert np.mean(moved) <= SHARE, n


# A key that is infinite, no number, or (f32) past what its first part can hold, among earlier positions and at the last of them.
# A query whose scores of it are -infinity has a result (weight 0), which a sum of parts alone turns into inf - inf.
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("value", [np.inf, -np.inf, 3.4e38, np.nan])
@pytest.mark.parametrize("cut,n", [(70, 75), (33, 40), (64, 700)])
def test_keys_that_are_no_numbers(dev, f16, value, cut, n):
    if f16 and value == 3.4e38:
        pytest.skip("no such half")
    heads, hd, max_pos = 4, 64, 800
    model = mirror(dev, heads, heads, hd, max_pos, 1.0, 1.0)
    if f16:
        model.set_kv_f16(True)
    tokens = [int(t) for t in np.random.default_rng(cut).integers(0, 256, cut + n)]
    model.prefill(tokens[:cut], 0, want_logits=False)
    dt = np.float16 if f16 else np.float32
    k_ptr, _, _ = model.kv_cache()
    for pos, d, x in ((5, 3, value), (cut - 1, 40, value)):
        if pos == 5 and n == 75:
            continue  # one alone
        a = np.array([x], dt)
        hip._check(hip.lib().candy_hip_h2d(dev.handle, k_ptr + ((2 * max_pos + pos) * hd + d) * a.itemsize, a.ctypes.data, a.nbytes))
    want, got = both(dev, model, tokens[cut:], cut)
    has = np.all(np.isfinite(want), axis=1)
    assert np.isnan(value) or 0.1 < np.mean(has) < 0.9
    assert np.all(np.isfinite(got[has]))
    if np.any(has):
        w, g = want[has].reshape(-1, 32), got[has].reshape(-1, 32)
        assert np.mean(np.abs(g - w) > 0.5 * np.max(np.abs(w), axis=1, keepdims=True) / 127) <= 2 * SHARE


# The same behind a query that has no result: its row stays no number, also where the attention kernel quantizes it by itself
# (from 256 rows on).
@pytest.mark.parametrize("heads,head_dim", [(4, 64), (2, 128)])
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("n", [40, 300])
def test_rows_without_a_number_stay_so(dev, heads, head_dim, f16, n):
    max_pos = 400
    model = mirror(dev, heads, heads, head_dim, max_pos, 1.0, 1.0)
    if f16:
        model.set_kv_f16(True)
    tokens = [int(t) for t in np.random.default_rng(n).integers(0, 256, 64 + n)]
    model.prefill(tokens[:64], 0, want_logits=False)
    a = np.array([np.nan], np.float16 if f16 else np.float32)
    hip._check(hip.lib().candy_hip_h2d(dev.handle, model.kv_cache()[0] + 5 * head_dim * a.itemsize, a.ctypes.data, a.nbytes))
    for rows in both(dev, model, tokens[64:], 64):
        assert not np.any(np.isfinite(rows[:, :head_dim]))


# No memory for the parts of K and V: the prompt is taken all the same, by the vector kernel, and the next one with memory by the
# matrix cores.  Positions in front that were cached either way serve both.
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("n", [40, 300])
def test_prompt_without_memory_for_parts(dev, head_dim, n):
    model = mirror(dev, 256 // head_dim, 256 // head_dim, head_dim, 4096, 1.0, 1.0)  # parts of 8 to 12 MB
    tokens = [int(t) for t in np.random.default_rng(n).integers(0, 256, n)]

    def rows(option, value, cut):
        """Hidden rows of the last pass; the option is set for the first one."""
        dev.set_option(option, value)
        try:
            model.prefill(tokens[:cut], 0, want_logits=False)
        finally:
            dev.set_option(option, 0)
        if cut < n:
            model.prefill(tokens[cut:], cut, want_logits=False)
        return model.prompt_hidden(n if cut == n else n - cut)

    for cut in (n, 33):
        want = rows("prefill.attention_valu", 1, cut)
        assert np.array_equal(rows("prefill.kv_parts_mb", 1, cut), want)
        got = rows("prefill.kv_parts_mb", 0, cut)
        level = np.max(np.abs(want).reshape(len(want), -1, 32), axis=2, keepdims=True) / 127
        assert np.mean(np.abs(got - want).reshape(len(want), -1, 32) > 0.5 * level) <= SHARE, cut


# The parts of earlier positions come out of the rope launch, or (split sums not folded) out of one of their own: the same bits.
# Those positions are cached by decode steps here, so that the parts an earlier prompt left are another sequence's.
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(8, 2, 64), (4, 2, 128)])
@pytest.mark.parametrize("cut,n", [(1, 2), (33, 40), (70, 3)])
def test_parts_of_earlier_positions(dev, heads, kv_heads, head_dim, cut, n):
    model = mirror(dev, heads, kv_heads, head_dim, 300, 1.0, 1.0)
    tokens = [int(t) for t in np.random.default_rng(cut).integers(0, 256, cut + n)]
    model.prefill(tokens[::-1], 0, want_logits=False)
    for p in range(cut):
        model.decode(tokens[p], p, want_logits=False)
    want, got = both(dev, model, tokens[cut:], cut)
    level = np.max(np.abs(want).reshape(n, -1, 32), axis=2, keepdims=True) / 127
    assert np.mean(np.abs(got - want).reshape(n, -1, 32) > 0.5 * level) <= max(SHARE, 2 / want.size)
    model.prefill(tokens[::-1], 0, want_logits=False)
    for p in range(cut):
        model.decode(tokens[p], p, want_logits=False)
    dev.set_option("prefill.fold_split_sums", 0)
    try:
        model.prefill(tokens[cut:], cut, want_logits=False)
        assert np.array_equal(model.prompt_hidden(n), got)
    finally:
        dev.set_option("prefill.fold_split_sums", 1)
