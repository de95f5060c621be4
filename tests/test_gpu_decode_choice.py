"""Decode steps that are asked for the greedy token and steps that are not (two captured graphs of one model), in turns."""
import ctypes

import numpy as np
import pytest

from candy_amd import gulisun, hip
from tests import gulisun_models as gm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [True, False])
def test_steps_with_and_without_the_greedy_token(graph):
    dev = hip.Device(0)
    cfg = gm.CONFIGS["odd"]
    w = gm.weights(cfg, seed=3, steady=True)
    L, V = hip.lib(), cfg["vocab"]

    def fresh():
        m = gulisun.build(dev, cfg, gm.Tensors(w), 32, hip.ACT_BF16)
        m.set_graph(graph)
        return m

    def step(m, token, pos, ask):
        nt = ctypes.c_int32(-7)
        p = ctypes.c_void_p()
        hip._check(L.candy_hip_decoder_decode(m.handle, token, pos, ctypes.byref(p), ctypes.byref(nt) if ask else None))
        out = np.empty(V, np.float32)
        hip._check(L.candy_hip_d2h(dev.handle, out.ctypes.data, p, out.nbytes))
        return out, nt.value

    tokens = [int(t) for t in np.random.default_rng(4).integers(0, V, 10)]
    always, sometimes = fresh(), fresh()
    for pos, t in enumerate(tokens):
        want, chosen = step(always, t, pos, True)
        got, token = step(sometimes, t, pos, pos % 3 == 2)
        assert chosen == int(np.argmax(want))
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) and token == (chosen if pos % 3 == 2 else -7)
    # greedy generation needs every step's choice, whatever the steps in front of it asked for
    n = 6
    a = (ctypes.c_int32 * n)()
    hip._check(L.candy_hip_decoder_generate(always.handle, 5, len(tokens), n, a))
    step_tokens, t = [], 5
    for i in range(n):
        _, t = step(sometimes, t, len(tokens) + i, True)
        step_tokens.append(t)
    assert list(a) == step_tokens
    # a prompt that asks, behind one that does not
    ids = (ctypes.c_int32 * 4)(*tokens[:4])
    p, nt = ctypes.c_void_p(), ctypes.c_int32(-7)
    hip._check(L.candy_hip_decoder_prefill(always.handle, ids, 4, 0, ctypes.byref(p), None))
    out = np.empty(V, np.float32)
    hip._check(L.candy_hip_d2h(dev.handle, out.ctypes.data, p, out.nbytes))
    hip._check(L.candy_hip_decoder_prefill(always.handle, ids, 4, 0, ctypes.byref(p), ctypes.byref(nt)))
    assert nt.value == int(np.argmax(out))
    always.free()
    sometimes.free()
    dev.close()
