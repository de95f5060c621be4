"""Grids of fp16 tiles whose last round is split along K: against the oracle, and against tiles that are all whole."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o

LIB = ctypes.CDLL(hip.LIB_PATH)
OTHERS = [synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML]  # one rule for all but Q4_K


def plan(fmt, rows, cols, m, deferred=0, cus=256):
    """Tile, tiles of it, how many are whole, and the lengths of the others' parts in super-blocks."""
    out = (ctypes.c_int * 5)()
    code = LIB.candy_test_f16_tail(fmt, (ctypes.c_int64 * len(rows))(*rows), len(rows), ctypes.c_int64(cols), ctypes.c_int64(m), cus, deferred, out)
    tiles, whole, splits, sb, _ = out
    return divmod(code, 1000), tiles, whole, [min(sb, cols // 256 - k * sb) for k in range(splits)]


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


def parts(n, sb, last):
    return [sb] * (n - 1) + [last]


# Tiles, tiles of the last round and their parts: two, three, more, the most there are; of equal length, a last one that is shorter, one
# super-block of it; weight rows that end inside a tile and not at a multiple of four; one activation row in the last column, and all
Q4K_CASES = [
    (16912, 3328, 195, (112, 128), 46, parts(5, 3, 1)), (20048, 3328, 200, (112, 128), 102, parts(2, 7, 6)),
    (17024, 2304, 288, (112, 192), 48, parts(3, 3, 3)), (17472, 3328, 277, (112, 192), 56, parts(4, 4, 1)),
    (8400, 2816, 822, (112, 256), 44, parts(4, 3, 2)), (7280, 4352, 1025, (112, 256), 69, parts(3, 6, 5)),
    (8960, 11008, 771, (112, 256), 64, parts(4, 11, 10)),
    (16512, 2048, 194, (128, 128), 2, parts(4, 2, 2)), (22121, 3328, 193, (128, 128), 90, parts(2, 7, 6)), (33000, 2304, 100, (128, 128), 2, parts(3, 3, 3)),
    (33641, 2816, 130, (128, 192), 7, parts(4, 3, 2)), (16685, 4864, 305, (128, 192), 6, parts(7, 3, 1)), (11008, 11008, 513, (128, 192), 2, parts(15, 3, 1)),
    (11008, 2048, 700, (128, 256), 2, parts(4, 2, 2)), (10301, 3584, 799, (128, 256), 68, parts(3, 5, 4)),
    (32770, 2048, 200, (128, 256), 1, parts(4, 2, 2)), (4736, 11776, 1538, (128, 256), 3, parts(16, 3, 1))]
OTHER_CASES = [
    (33000, 2304, 100, (128, 128), 2, parts(3, 3, 3)),
    (10985, 2048, 513, (128, 192), 2, parts(4, 2, 2)), (6045, 2560, 1339, (128, 192), 80, parts(3, 4, 2)), (17024, 3328, 277, (128, 192), 10, parts(5, 3, 1)),
    (21951, 3328, 289, (128, 192), 88, parts(2, 7, 6)),
    (32770, 2048, 200, (128, 256), 1, parts(4, 2, 2)), (11008, 2048, 1400, (128, 256), 4, parts(4, 2, 2)), (8733, 6400, 1026, (128, 256), 89, parts(2, 13, 12)),
    (8320, 4352, 796, (128, 256), 4, parts(6, 3, 2)), (4704, 6400, 1556, (128, 256), 3, parts(9, 3, 1))]
CASES = [(synth.Q4_K, *c) for c in Q4K_CASES] + [(f, *c) for c in OTHER_CASES for f in OTHERS]


@pytest.mark.parametrize("fmt,rows,cols,m,tile,last_round,lengths", CASES)
def test_the_plan_of_each_case(fmt, rows, cols, m, tile, last_round, lengths):
    got, tiles, whole_tiles, split = plan(fmt, (rows,), cols, m)
    assert (got, tiles - whole_tiles, split) == (tile, last_round, lengths)


def test_every_part_has_work_and_the_round_has_room():
    rng = np.random.default_rng(7)
    seen = 0
    for _ in range(40000):
        fmt, cus = int(rng.choice([synth.Q4_K, synth.Q6_K])), int(rng.choice([64, 256, 304]))
        rows, cols, m = (int(rng.integers(1, 40000)),), 256 * int(rng.integers(1, 60)), int(rng.integers(33, 2100))
        _, tiles, whole_tiles, split = plan(fmt, rows, cols, m, cus=cus)
        if split:
            seen += 1
            assert whole_tiles % cus == 0 and 0 < tiles - whole_tiles <= cus // 2 and (tiles - whole_tiles) * len(split) <= cus
            assert sum(split) == cols // 256 and min(split) > 0 and 2 <= len(split) <= 16
        else:
            assert whole_tiles == tiles
    assert seen > 500


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,rows,cols,m,tile,last_round,lengths", CASES)
def test_last_round_in_splits(dev, fmt, rows, cols, m, tile, last_round, lengths):
    w = synth.random_weight(fmt, rows, cols, seed=rows + fmt)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    got = dev.qmatmul(q, x)
    want = whole(dev, lambda: dev.qmatmul(q, x))
    # the same products in sums of another order, and only in the last round's tiles: a few 2^-24 of sums of 2048 values, and of longer ones
    # as the root of their length
    assert np.max(np.abs(got - want)) <= max(2e-6, cols ** 0.5 * 2.0 ** -24) * np.max(np.abs(want))
    moved = np.any(got != want, axis=0)
    n_tiles = -(-rows // tile[0])
    first = max(0, n_tiles - last_round) * tile[0]  # of the last column of tiles, or of all of it and more
    assert np.any(moved) and not np.any(moved[:first])
    q.free()
    sub, some = np.unique(np.r_[0:rows:499, rows - 130:rows]), np.unique(np.r_[0, 191, 192, 255, 256, 511, 512, m - 1])
    some = some[some < m]
    part = np.ascontiguousarray(w.reshape(rows, -1)[sub]).reshape(-1)
    want = o.qmatmul(fmt, part, len(sub), cols, x[some])
    # weight and activation of a product are each rounded to fp16, by up to 2^-11 of it and evenly within that: sqrt(2 / 3) 2^-11 of the
    # root of the products' sum of squares; six times that for the largest of some thousand
    values = o.dequantize(fmt, part).reshape(len(sub), cols).astype(np.float64)
    spread = np.sqrt((x[some].astype(np.float64) ** 2) @ (values ** 2).T) * (2 / 3) ** 0.5 * 2.0 ** -11
    assert np.all(np.abs(got[some][:, sub] - want) <= 6 * spread)


@pytest.mark.gpu
def test_three_tensors_and_a_residual(dev):
    """A prompt whose q / k / v (one grid, tiles of the last round in two of the tensors) and o (with the residual) end in splits."""
    n, d = 2100, 4096
    assert plan(synth.Q4_K, (d, d, d), d, n, deferred=1) == ((128, 256), 864, 768, [8, 8]) and plan(synth.Q4_K, (d,), d, n, 1)[1:] == (288, 256, [2] * 8)
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
