"""The contraction that deals K to wavefronts as the prompt pass launches it: several weights on a grid, residuals in the epilogue, odd
numbers of weight rows; and its operands as the norm and SiLU launches write them."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth
from oracle import oracle as o

pytestmark = pytest.mark.gpu
LIB = ctypes.CDLL(hip.LIB_PATH)
P = ctypes.c_void_p
LIB.candy_test_rows_launch.argtypes = [P, ctypes.c_int, P, P, P, P, ctypes.c_int64]
LIB.candy_test_rows_image.argtypes = [P, ctypes.c_int, P, P, ctypes.c_int64, ctypes.c_int64, P, P, P]


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def launch(dev, ws, ys, res, x):
    arr = lambda ps: (P * len(ps))(*ps)
    src = dev.from_numpy(x)
    hip._check(LIB.candy_test_rows_launch(dev.handle, len(ws), arr([w.handle for w in ws]), arr([y.ptr for y in ys]),
                                          arr([r.ptr if r else None for r in res]), src.ptr, len(x)))
    return [y.download(np.float32, len(x) * w.rows).reshape(len(x), w.rows) for y, w in zip(ys, ws)]


# Weight rows off the strips of 16, off the float4 stores and under two strips; batches of every tile height
@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.Q4_0, synth.Q4_0_GGML])
@pytest.mark.parametrize("m", [3, 16, 20, 40, 50, 100, 255])
def test_weights_that_share_a_launch_and_residuals(dev, fmt, m):
    cols, rows = 1024, (131, 17, 1002)
    blocks = [synth.random_weight(fmt, r, cols, seed=fmt + r) for r in rows]
    ws = [dev.qtensor(fmt, r, cols, b) for r, b in zip(rows, blocks)]
    x = synth.random_activations(m, cols, seed=m)
    new = lambda: [dev.alloc(4 * m * r) for r in rows]
    alone = [launch(dev, [w], [y], [None], x)[0] for w, y in zip(ws, new())]
    sub = np.unique(np.r_[0, m // 2, m - 1])
    for a, b, r in zip(alone, blocks, rows):
        want = o.qmatmul(fmt, b, r, cols, x[sub])
        assert np.max(np.abs(a[sub] - want)) <= 2e-5 * np.max(np.abs(want))
    near = lambda a, b, more=0.0: np.max(np.abs(a - b)) <= 2e-6 * (np.max(np.abs(b)) + more)  # 8 or 16 wavefronts: two orders of f32 sums
    assert all(near(a, b) for a, b in zip(launch(dev, ws, new(), [None] * 3, x), alone))
    # a residual of its own, one that is the output, none
    h = [np.random.default_rng(r).standard_normal((m, r)).astype(np.float32) for r in rows]
    ys, other = new(), dev.from_numpy(h[0])
    ys[1].upload(h[1])
    got = launch(dev, ws, ys, [other, ys[1], None], x)
    for g, a, r in zip(got, alone, (h[0], h[1], 0)):
        assert near(g, a + r, np.max(np.abs(a)))
    assert np.array_equal(other.download(np.float32, m * rows[0]).reshape(m, -1), h[0])


# Norms of one row in registers (4096, 8192 values) and of any length; one, three and sixteen tiles of 16 rows
@pytest.mark.parametrize("silu", [0, 1])
@pytest.mark.parametrize("m,cols", [(3, 256), (17, 4096), (40, 4352), (5, 8192), (9, 8448), (255, 512)])
def test_operands_as_the_launch_in_front_writes_them(dev, silu, m, cols):
    rng = np.random.default_rng(m + cols)
    a = rng.standard_normal((m, cols)).astype(np.float32)
    b = rng.standard_normal((m, cols) if silu else cols).astype(np.float32)
    a[0, 32:64] = 0  # an empty block
    tiles = (m + 15) // 16 if m <= 48 else (m + 63) // 64 * 4
    frag_bytes = (16 * cols + 255) // 256 * 256
    scale_bytes = ((cols // 256 + 1) * 512 + 255) // 256 * 256
    image, qs, sc = dev.alloc(tiles * (frag_bytes + 2 * scale_bytes)), dev.alloc(m * cols), dev.alloc(m * cols // 32 * 8)
    hip._check(LIB.candy_test_rows_image(dev.handle, silu, dev.from_numpy(a).ptr, dev.from_numpy(b).ptr, m, cols, image.ptr, qs.ptr, sc.ptr))
    raw = image.download(np.uint8, image.nbytes)
    q = qs.download(np.int8, m * cols).reshape(m, cols)
    s = sc.download(np.dtype([("d", np.float32), ("sum", np.int32)]), m * cols // 32).reshape(m, cols // 32)
    assert q.any()
    frag = raw[:tiles * frag_bytes].reshape(tiles, frag_bytes)[:, :16 * cols].view(np.int8)
    # [tile][super-block][pair][chunk][row][sub-block of the pair][8 values] -> [row][super-block, pair, sub-block, chunk, value]
    f = frag.reshape(tiles, cols // 256, 4, 4, 16, 2, 8).transpose(0, 4, 1, 2, 5, 3, 6).reshape(16 * tiles, cols)
    assert np.array_equal(f[:m], q)
    at = tiles * frag_bytes
    for values in (s["d"], s["d"] * s["sum"].astype(np.float32)):
        t = raw[at:at + tiles * scale_bytes].reshape(tiles, scale_bytes)[:, :cols // 256 * 512].copy().view(np.float32)
        t = t.reshape(tiles, cols // 256, 16, 8).transpose(0, 2, 1, 3).reshape(16 * tiles, cols // 32)
        assert np.array_equal(t[:m].view(np.uint32), values.view(np.uint32))
        at += tiles * scale_bytes
