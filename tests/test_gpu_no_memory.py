"""Calls that need memory only to be faster are answered without it."""
import ctypes

import numpy as np
import pytest

from candy_amd import hip, synth

pytestmark = pytest.mark.gpu
LIB = ctypes.CDLL(hip.LIB_PATH)
LIB.candy_test_fail_alloc.argtypes = [ctypes.c_void_p, ctypes.c_int]
LIB.candy_test_fail_alloc.restype = None


@pytest.fixture
def dev():
    d = hip.Device(0)
    yield d
    LIB.candy_test_fail_alloc(d.handle, 0)
    d.close()


@pytest.mark.parametrize("fmt,rows,cols,m", [(synth.Q5_K, 8192, 4096, 6), (synth.Q6_K, 4112, 4096, 15)])
def test_planar_quants_without_memory_for_their_order(dev, fmt, rows, cols, m):
    """Fewer than 16 rows: the vector kernels and the unsplit tiles take no device memory."""
    L, act = hip.lib(), ctypes.c_void_p()
    w = dev.qtensor(fmt, rows, cols, synth.random_weight(fmt, rows, cols, seed=fmt))
    x = synth.random_activations(m, cols, seed=m)
    src, dst = dev.from_numpy(x), dev.alloc(4 * m * rows)
    hip._check(L.candy_hip_qact_create(dev.handle, m, cols, ctypes.byref(act)))
    hip._check(L.candy_hip_qact_quantize(act, src.ptr, m, cols))

    def call():
        hip._check(L.candy_hip_qmatmul_qact(dev.handle, w.handle, act, dst.ptr))
        return dst.download(np.float32, m * rows)

    assert dev.get_option("runtime.workspace_bytes") == 0
    LIB.candy_test_fail_alloc(dev.handle, 1)
    got = call()
    dev.set_option("rows.i8", 0)
    want = call()
    dev.set_option("rows.i8", 1)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert np.max(np.abs(call() - want)) <= 2e-6 * np.max(np.abs(want))  # with memory again: another order of f32 sums
    assert dev.get_option("runtime.workspace_bytes") > 0
    hip._check(L.candy_hip_qact_free(act))
