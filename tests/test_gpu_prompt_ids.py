"""Every token of a prompt reaches its row, whatever the launches or the copy that brought it: a window of one position, so that a row
depends on its own token alone."""
import numpy as np
import pytest

from candy_amd import hip, suvazen
from tests import suvazen_models as sm

pytestmark = pytest.mark.gpu


# one launch and two of 960 tokens, a full last one, and past sixteen of them, where the tokens are copied
@pytest.mark.parametrize("n", [959, 960, 961, 1920, 15360, 15361])
def test_rows_go_by_their_tokens(n):
    dev = hip.Device(0)
    cfg = sm.config([(sm.mixer(2, 1, 32, window=1), 64)], width=64, vocab=173)
    m = suvazen.build(dev, cfg, sm.Tensors(sm.weights(cfg, seed=1)), 15361, hip.ACT_F32)
    V = cfg["vocab"]
    m.prefill(range(V), 0, want_logits=False)
    table = m.prompt_hidden(V)
    tokens = np.random.default_rng(n).integers(0, V, n)
    m.prefill(tokens, 0, want_logits=False)
    got = m.prompt_hidden(n)
    # a few f32 sums in another order (other tiles); another token's row is another row
    assert np.max(np.abs(got - table[tokens])) <= 1e-4 * np.max(np.abs(table))
    m.free()
    dev.close()
