"""Prompt attention over latents whose keys and values go to LDS by direct loads: heads of 64 and 128 values with 33 to 64 rotated ones."""
import numpy as np
import pytest

from candy_amd import hip
from tests import gulisun_models as gm
from tests.test_gpu_gulisun import Latent
from tests.test_gpu_suvazen import rel

pytestmark = pytest.mark.gpu

# against the oracle, which leaves the rebuilt keys and values unrounded: results in bfloat16 (2^-9 of each) and operands rounded to it
# (2^-8 of a few), summed over a row
TOL = 1.5e-2


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def transposed(dev, call):
    """The kernel that moves values to LDS transposed: the same products in the same order."""
    dev.set_option("prefill.latent_direct", 0)
    try:
        return call()
    finally:
        dev.set_option("prefill.latent_direct", 1)


def same_bits(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


# rotated halves of whole eights and not; one tile and a row, tiles cut short in front of and behind the portion's start
@pytest.mark.parametrize("heads,dim,rot,vdim", [(2, 64, 64, 64), (3, 64, 62, 128), (2, 128, 40, 64), (1, 128, 48, 128), (5, 120, 64, 100)])
def test_portions(dev, heads, dim, rot, vdim):
    n = 131
    case = Latent(dev, gm.latent(heads, dim, rot, vdim, 96, 40, 500.0, None)["mixer"], n, heads + rot)
    sink = np.random.default_rng(rot).standard_normal(heads).astype(np.float32)
    for s in (sink, None):
        want = case.oracle(s, hip.ACT_BF16)
        for portions in ([n], [2, 62, 67], [64, 2, 65], [63, 68], [129, 2]):
            got = case.device(s, hip.ACT_BF16, portions)
            assert rel(got, want) < TOL, (s is None, portions)
            assert same_bits(got, transposed(dev, lambda: case.device(s, hip.ACT_BF16, portions))), (s is None, portions)


# more workgroups than CUs, the rest of them in the other order: every block of queries is somebody's
@pytest.mark.parametrize("heads,n", [(16, 1030), (16, 2048), (32, 1000)])
def test_order_of_the_blocks(dev, heads, n):
    case = Latent(dev, gm.latent(heads, 64, 64, 64, 64, 32, 500.0, None)["mixer"], n, n)
    want = case.oracle(None, hip.ACT_BF16)
    got = case.device(None, hip.ACT_BF16, [n])
    assert rel(got, want) < TOL
    assert same_bits(got, transposed(dev, lambda: case.device(None, hip.ACT_BF16, [n])))
