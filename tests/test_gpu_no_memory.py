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


def test_prompt_without_memory_for_its_operands(dev):
    """Of a prompt's buffers one may be missing: the operands of the exact kernel.  Without it the tiles take the prompt."""
    c = dict(n_layers=2, d_model=512, n_heads=4, n_kv_heads=2, head_dim=128, d_ffn=1024, vocab=256, max_pos=64, rms_eps=1e-5, rope_base=10000.0)
    kinds = {hip.W_Q: (512, 512), hip.W_K: (256, 512), hip.W_V: (256, 512), hip.W_O: (512, 512), hip.W_GATE: (1024, 512), hip.W_UP: (1024, 512),
             hip.W_DOWN: (512, 1024)}
    draw = lambda fmt, r, k, seed: dev.qtensor(fmt, r, k, synth.random_weight(fmt, r, k, seed=seed, scale=synth.unit_scale(fmt)))
    weights = [(kind, l, draw(synth.Q4_K, *shape, 7 * l + kind)) for l in range(2) for kind, shape in kinds.items()] + \
              [(kind, -1, draw(synth.Q8_0, 256, 512, 50 + kind)) for kind in (hip.W_HEAD, hip.W_EMBED)]
    tokens = [int(t) for t in np.random.default_rng(1).integers(0, 256, 20)]

    def model():
        m = hip.Llama(dev, **c)
        for kind, l, w in weights:
            m.set_qweight(kind, l, w)
        for kind, l in ((hip.W_ATTN_NORM, 0), (hip.W_FFN_NORM, 0), (hip.W_ATTN_NORM, 1), (hip.W_FFN_NORM, 1), (hip.W_OUT_NORM, -1)):
            m.set_norm(kind, l, np.ones(512, np.float32))
        m.set_kv_f16(True)
        return m

    def rows(nth=0):
        m = model()
        LIB.candy_test_fail_alloc(dev.handle, nth)
        try:
            m.prefill(tokens, 0, want_logits=False)
        except hip.CandyHipError:
            return None
        finally:
            LIB.candy_test_fail_alloc(dev.handle, 0)
        out = m.prompt_hidden(20)
        m.prefill(tokens[:9], 0, want_logits=False)  # the next, shorter prompt finds it missing too
        return out, m.prompt_hidden(9)

    exact = rows()
    dev.set_option("rows.i8", 0)
    tiles = rows()
    dev.set_option("rows.i8", 1)
    same = lambda a, b: all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(a, b))
    assert not same(exact, tiles)
    got = [rows(nth) for nth in range(1, 30)]
    answered = [nth for nth, g in enumerate(got) if g and not same(g, exact)]
    assert len(answered) == 1 and same(got[answered[0]], tiles)
    assert got[0] is None and same(got[-1], exact)


@pytest.mark.parametrize("fmt,rows,cols,m", [(synth.Q4_K, 11008, 2048, 700), (synth.Q8_0, 21951, 3328, 289)])
def test_tiles_without_memory_for_the_parts_of_their_last_round(dev, fmt, rows, cols, m):
    """Grids whose last round is split along K: without the workspace its tiles stay whole."""
    L = hip.lib()
    w = dev.qtensor(fmt, rows, cols, synth.random_weight(fmt, rows, cols, seed=m))
    src, dst = dev.from_numpy(synth.random_activations(m, cols, seed=rows)), dev.alloc(4 * m * rows)

    def call():
        hip._check(L.candy_hip_qmatmul(dev.handle, w.handle, src.ptr, m, dst.ptr))
        return dst.download(np.float32, m * rows)

    dev.set_option("mmq.f16_split", 1)
    whole = call()
    dev.set_option("mmq.f16_split", 0)
    assert dev.get_option("runtime.split_workspace_bytes") == 0
    LIB.candy_test_fail_alloc(dev.handle, 1)
    assert np.array_equal(call().view(np.uint32), whole.view(np.uint32))
    assert dev.get_option("runtime.split_workspace_bytes") == 0
    got = call()  # with memory again: sums in another order
    assert dev.get_option("runtime.split_workspace_bytes") > 0 and np.any(got != whole)
    assert np.max(np.abs(got - whole)) <= max(2e-6, cols ** 0.5 * 2.0 ** -24) * np.max(np.abs(whole))


@pytest.mark.parametrize("fmt,rows,m,mib", [(synth.Q4_1, 64, 100, 5), (synth.Q4_K, 512, 8, 1), (synth.Q8_0, 4096, 40, 1)])
def test_the_workspace_holds_what_the_call_uses(dev, fmt, rows, m, mib):
    """Quants, their fp16 image and operands only where the kernel that runs reads them (8192 values a row, in whole MiB)."""
    cols = 8192
    w = dev.qtensor(fmt, rows, cols, synth.random_weight(fmt, rows, cols, seed=fmt))
    dev.qmatmul(w, synth.random_activations(m, cols, seed=m))
    assert dev.get_option("runtime.workspace_bytes") == mib << 20
