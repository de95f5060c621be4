"""fp16 contraction of up to 128 activation rows with K dealt to the wavefronts, against the 128 x 128 tiles on the same fp16
operands and against the oracle: every kernel that the library's rule can choose."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o

FORMATS = [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML]
FRAGMENTS = {3: (33, 48), 4: (49, 64), 5: (65, 80), 6: (81, 96), 7: (97, 112), 8: (113, 128)}  # of 16 activation rows: first and last count
WEIGHT_ROWS = {1: (2048, 4096), 2: (4097, 8192), 3: (8193, 12288)}              # fragments of 16 weight rows on 256 CUs

LIB = ctypes.CDLL(hip.LIB_PATH)
LIB.candy_test_rows_fragments.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_int]


def chosen(fmt, m, rows, cols, cus=256):
    """Weight fragments per workgroup, 0: the tiles."""
    return LIB.candy_test_rows_fragments(fmt, rows, cols, m, cus)


def fragments(m):
    return next(f for f, (_, last) in FRAGMENTS.items() if m <= last)


def shapes():
    """Per kernel: the fewest rows on either side with as many super-blocks as the rule allows, and the most rows (less one
    weight row, a length not in fours) with as few of them."""
    for fmt in FORMATS:
        for rf, (few, most) in WEIGHT_ROWS.items():
            for mf, (low, high) in FRAGMENTS.items():
                lengths = range(256, 12800, 256)
                for m, rows, pick in ((low, few + 1, max), (high, most - 1, min)):
                    cols = pick((c for c in lengths if chosen(fmt, m, rows, c) == rf), default=0)
                    if cols:
                        yield fmt, rf, mf, m, rows, cols


SHAPES = list(shapes())


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,rf,mf,m,rows,cols", SHAPES)
def test_rows_against_tiles_and_oracle(dev, fmt, rf, mf, m, rows, cols):
    assert chosen(fmt, m, rows, cols) == rf and fragments(m) == mf
    w = synth.random_weight(fmt, rows, cols, seed=rows + m)
    x = synth.random_activations(m, cols, seed=cols + m)
    q = dev.qtensor(fmt, rows, cols, w)
    got = dev.qmatmul(q, x)
    assert np.array_equal(got.view(np.uint32), dev.qmatmul(q, x).view(np.uint32))
    dev.set_option("mmq.f16_shape", 2)
    try:
        tiles = dev.qmatmul(q, x)
    finally:
        dev.set_option("mmq.f16_shape", 0)
    top = np.max(np.abs(tiles))
    assert cols == 256 or not np.array_equal(got, tiles)  # two kernels: another order of the sums (of a single super-block the same)
    # the same products in another order: K sums of f32, 2^-24 each of a partial sum no larger than the largest result's
    # order (random signs: sqrt(K) of them, 64 * 2^-24 = 4e-6 at K = 4096)
    assert np.max(np.abs(got - tiles)) <= max(cols, 4096) ** 0.5 * 2.0 ** -24 * 1.05 * top
    sub = np.unique(np.r_[0:rows:97, rows - 17:rows])
    nb = synth.weight_nbytes(fmt, 1, cols)
    want = o.qmatmul(fmt, w.reshape(rows, nb)[sub].reshape(-1), len(sub), cols, x)
    # fp16 operands: 2^-12 of each product, as for the tiles
    assert np.max(np.abs(got[:, sub] - want)) <= 5e-4 * np.max(np.abs(want))


# ------------------------------------------------------------------ the rule, on the CPU
def test_fragments_of_a_batch():
    assert all(LIB.candy_test_rows_activation_fragments(ctypes.c_int64(m)) == fragments(m) for m in range(33, 129))


def test_one_round_of_workgroups_and_bounded_activations():
    rng = np.random.default_rng(5)
    seen = set()
    for _ in range(20000):
        fmt, m = int(rng.choice(FORMATS)), int(rng.integers(1, 140))
        rows, cols, cus = int(2 ** rng.uniform(8, 15)), 256 * int(2 ** rng.uniform(0, 6)), int(rng.choice([64, 256, 304]))
        rf = chosen(fmt, m, rows, cols, cus)
        assert 0 <= rf <= 3
        if rf:
            assert m <= 128 and rows >= 2048 and -(-rows // (16 * rf)) <= cus
            assert m > 64 or fmt in (synth.Q4_K, synth.Q6_K)
            assert (8 if m > 96 else fragments(m)) * 32 * cols <= 1.2e6  # seven are weighed as eight
            seen.add((fmt, rf, fragments(m)))
    assert seen == {s[:3] for s in SHAPES}  # no kernel but those tested above


@pytest.mark.parametrize("fmt,m,rows,cols,rf", [
    (synth.Q8_0, 77, 11008, 4096, 3), (synth.Q8_0, 128, 2048, 1024, 1), (synth.Q4_K, 80, 4096, 4096, 1), (synth.Q4_K, 33, 4096, 5632, 1),
    (synth.Q6_K, 48, 11008, 4096, 3), (synth.Q6_K, 48, 8192, 4096, 2), (synth.Q6_K, 96, 8192, 2048, 2), (synth.Q6_K, 80, 4096, 2304, 1),
    (synth.Q8_0, 96, 4096, 2304, 1), (synth.Q4_0, 80, 12288, 2304, 3), (synth.Q4_K, 48, 4096, 512, 1),
    # where the tiles are ahead: long rows, too many of them
    (synth.Q8_0, 77, 4096, 14336, 0), (synth.Q8_0, 77, 14336, 4096, 0), (synth.Q8_0, 129, 4096, 1024, 0), (synth.Q8_0, 64, 4096, 1024, 0),
    # rounds that most wavefronts sit out and odd rows of Q6_K, where the tiles were ahead before blocks came through LDS and a step's loads
    # stood in front of its arithmetic: us, tiles / rows, 23.4 / 17.1, 23.1 / 16.1, 18.2 / 15.4, 17.2 / 15.1, 18.3 / 16.2
    (synth.Q6_K, 64, 8200, 3328, 3), (synth.Q6_K, 48, 8200, 3840, 3), (synth.Q5_K, 128, 8192, 2304, 2), (synth.Q4_K, 128, 8192, 2304, 2),
    (synth.Q4_K, 80, 4200, 4352, 2)])
def test_where_the_lines_lie(fmt, m, rows, cols, rf):
    assert chosen(fmt, m, rows, cols) == rf


@pytest.mark.parametrize("fmt,m,rows,cols,rf", [
    # ahead of the tiles since a step's loads stand in front of its arithmetic (14.5 / 20.9 us, 7.8 / 11.1, 21.2 / 24.6, 24.1 / 26.7)
    (synth.Q4_K, 96, 8200, 2560, 3), (synth.Q5_K, 128, 4096, 512, 1), (synth.Q4_0, 128, 4096, 4096, 1), (synth.Q8_0, 128, 6144, 4096, 2),
    # one super-block in the last round: level with the tiles at eight fragments (21.4), ahead at five (18.7 / 16.2)
    (synth.Q5_K, 128, 4352, 4352, 0), (synth.Q4_K, 80, 4576, 4352, 2), (synth.Q4_K, 80, 4577, 4352, 2), (synth.Q4_K, 64, 4200, 4352, 2),
    # long rows of few weight rows and Q4_0 from 65 rows
    (synth.Q8_0, 96, 2816, 5632, 0), (synth.Q4_0, 66, 4096, 4096, 1),
    # Q6_K through LDS: three weight fragments beside five and six of activations, and odd blocks (8400 x 3328, 48 rows 22.1 / 15.7)
    (synth.Q6_K, 96, 11008, 4096, 3), (synth.Q6_K, 128, 8192, 4096, 2), (synth.Q6_K, 48, 8400, 3328, 3), (synth.Q6_K, 48, 8401, 3328, 3),
    (synth.Q6_K, 48, 8200, 2816, 3), (synth.Q6_K, 80, 8200, 3328, 3)])
def test_where_the_fitted_costs_cross(fmt, m, rows, cols, rf):
    assert chosen(fmt, m, rows, cols) == rf


@pytest.mark.parametrize("rows,cols,rf", [(8208, 2048, 3), (8208, 3072, 3), (10880, 3072, 3), (8208, 3328, 0), (8208, 4096, 0), (10752, 4096, 0),
                                          (10880, 4096, 0), (10881, 4096, 3), (10881, 3328, 3), (11008, 4096, 3), (12288, 4096, 3)])
def test_eight_fragments_of_q4_k_where_rows_are_short_or_the_tiles_many(rows, cols, rf):
    # the tiles are ahead where they share K by three (85 columns of them on 256 CUs at most) and rows are longer than 3072: us, 128 rows, tiles /
    # here 10880 x 4096 28.1 / 29.1, 8208 x 3328 24.8 / 25.4; 8208 x 3072 23.9 / 22.6, 10896 x 4096 31.1 / 29.1
    assert all(chosen(synth.Q4_K, m, rows, cols) == rf for m in (113, 120, 128))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,m", [(2049, 2304, 48), (2063, 256, 80), (4099, 2304, 64), (4111, 2048, 48), (8209, 1280, 48)])
def test_q6_k_blocks_behind_the_start_of_a_piece(dev, rows, cols, m):
    # odd rows of odd blocks start 2 .. 14 bytes into a piece, and the matrix ends in the middle of a word
    assert chosen(synth.Q6_K, m, rows, cols)
    w = synth.random_weight(synth.Q6_K, rows, cols, seed=rows)
    x = synth.random_activations(m, cols, seed=cols)
    got = dev.qmatmul(dev.qtensor(synth.Q6_K, rows, cols, w), x)
    nb = synth.weight_nbytes(synth.Q6_K, 1, cols)
    sub = np.r_[0:9, rows - 17:rows]
    want = o.qmatmul(synth.Q6_K, w.reshape(rows, nb)[sub].reshape(-1), len(sub), cols, x)
    # fp16 operands: 2^-12 of each product
    assert np.max(np.abs(got[:, sub] - want)) <= 5e-4 * np.max(np.abs(want))
