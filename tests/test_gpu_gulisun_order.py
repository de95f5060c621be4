"""A bfloat16 Gulisun prompt keeps the order of its sums: a last place that moves picks another expert at a near tie, and with it
another result row, so a faster tile or split is taken only where every bit stays.  The sums are the matrix instructions' own,
which no CPU restatement gives: the bits are those an MI355X gave with tiles of 128 x 128."""
import hashlib

import numpy as np
import pytest

from candy_amd import gulisun, hip
from tests import gulisun_models as gm

pytestmark = pytest.mark.gpu

# contractions that leave one, two and more copies of their sums; attention of widths in whole 64s and in between
CONFIG = gm.config([gm.latent(4, 128, 64, 128, 512, 1024, experts=8, top=3, ff=320, shared=1088),
                    gm.rglru(1024, 2, 4, experts=8, top=3, ff=320, shared=1088),
                    gm.latent(4, 128, 64, 128, 512, 1024, kv_from=0, experts=8, top=3, ff=320),
                    gm.latent(3, 64, 64, 64, 512, 520, sink=False, experts=8, top=3, ff=320, shared=512),
                    gm.latent(5, 56, 24, 72, 128, 200, experts=8, top=3, ff=320, shared=512)], 1024, 400)
BITS = {40: "308542761aa4ae64", 65: "36681a4ff68640c2", 200: "630f6477d594125a", 513: "75a0e93aadfa2a0d", 1100: "c358668f058bf8a0"}


def digests(dev):
    w = gm.weights(CONFIG, seed=7, peaky=1.5)
    m = gulisun.build(dev, CONFIG, gm.Tensors(w), 1104, hip.ACT_BF16)
    for n in sorted(BITS):
        tokens = [int(t) for t in np.random.default_rng(n).integers(0, CONFIG["vocab"], n)]
        _, logits = m.prefill(tokens, 0)
        yield n, hashlib.sha256(m.prompt_hidden(n).tobytes() + logits.tobytes()).hexdigest()[:16]
    m.free()


def test_bits_of_a_prompt():
    dev = hip.Device(0)
    assert dict(digests(dev)) == BITS
    dev.close()
