"""The norm chain of a decoder's layers with partial copies and expert slots: launches of few rows, which request them in batches,
give the bits of launches of many rows, which add them one by one; rows as wide as decoders have them, and ragged ones."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip

pytestmark = pytest.mark.gpu
LIB = ctypes.CDLL(hip.LIB_PATH)
LIB.candy_test_norm_chain.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_float, ctypes.c_float]
MANY, FEW, EPS, MULT = 600, 40, 1e-5, 0.75


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def norm(v, w, b, rms):
    v = v.astype(np.float64)
    if not rms:
        v = v - v.mean(1, keepdims=True)
    return v / np.sqrt((v * v).mean(1, keepdims=True) + EPS) * w + (0 if b is None else b)


# one, two and four float4 per thread, and eight (never in batches); copies of 8 + 4 + 2 + 1 and less; experts of 3, 6 and 9
@pytest.mark.parametrize("cols,copies,top", [(1000, 8, 0), (1030, 2, 0), (2048, 3, 6), (2048, 8, 0), (2100, 7, 3), (4096, 8, 9), (4090, 2, 0),
                                             (4096, 0, 6), (4034, 15, 0), (5000, 3, 3)])
@pytest.mark.parametrize("f32,rms,bias,ids", [(1, 0, 1, 0), (0, 1, 0, 0), (0, 0, 0, 1), (1, 1, 0, 1)])
def test_few_rows_and_many(dev, cols, copies, top, f32, rms, bias, ids):
    rng = np.random.default_rng(cols + copies)
    ld = (cols + 63) // 64 * 64

    def rows(n):  # padded with zeros
        a = np.zeros((n, ld), np.float32)
        a[:, :cols] = rng.standard_normal((n, cols)).astype(np.float32)
        return a

    x, y, slots = rows(MANY), [rows(MANY) for _ in range(copies)], rows(MANY * top)
    gate = rng.random(MANY * top).astype(np.float32)
    post_w, post_b, pre_w, pre_b, step = (rows(1) for _ in range(5))
    order = rng.permutation(MANY).astype(np.int32)
    keep = [dev.from_numpy(a) if a is not None and a.size else None
            for a in (x, np.stack(y) if y else None, slots, gate, post_w, post_b if bias else None, step, None, pre_w, pre_b if bias else None,
                      None, order if ids else None)]

    def run(n):
        x_out, out = dev.alloc(MANY * ld * 4), dev.alloc(MANY * ld * 4)
        hip._check(hip.lib().candy_hip_zero(dev.handle, out.ptr, out.nbytes))
        ptr = [b.ptr if b else None for b in keep]
        ptr[7], ptr[10] = x_out.ptr, out.ptr
        num = (ctypes.c_int64 * 11)(ld, ld, copies, MANY * ld, ld, top, ld, f32, rms, n, cols)
        hip._check(LIB.candy_test_norm_chain(dev.handle, (ctypes.c_void_p * 12)(*ptr), num, MULT, EPS))
        return x_out.download(np.uint32, n * ld).reshape(n, ld), out.download(np.uint32 if f32 else np.uint16, n * ld).reshape(n, ld)

    few, many = run(FEW), run(MANY)
    assert np.array_equal(few[0], many[0][:FEW]) and np.array_equal(few[1], many[1][:FEW])
    src = order[:FEW] if ids else np.arange(FEW)
    total = sum((c[src].astype(np.float64) for c in y), np.zeros((FEW, ld)))
    if top:
        picked = slots.reshape(MANY, top, ld)[src] * gate.reshape(MANY, top)[src][:, :, None].astype(np.float64)
        total = total + picked.sum(1)
    w = lambda a: a[0, :cols].astype(np.float64)
    want_x = x[src, :cols] + MULT * norm(total[:, :cols], w(post_w), w(post_b) if bias else None, rms) + w(step)
    got_x = few[0].view(np.float32)[:, :cols]
    assert np.max(np.abs(got_x - want_x)) <= 2e-5 * np.max(np.abs(want_x))
    want = norm(want_x, w(pre_w), w(pre_b) if bias else None, rms)
    got = few[1].view(np.float32)[:, :cols] if f32 else hip.bf16_values(few[1])[:, :cols]
    assert np.max(np.abs(got - want)) <= (2e-5 if f32 else 2.0 ** -8) * np.max(np.abs(want))
