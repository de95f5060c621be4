"""Rules of the expert layers' one-row kernels, on the CPU."""
import ctypes

import pytest

from candy_amd import hip

LIB = ctypes.CDLL(hip.LIB_PATH)


@pytest.mark.parametrize("cus", [64, 256, 304])
@pytest.mark.parametrize("shared", [0, 64, 2816])
def test_a_wavefront_that_reads_the_choice_has_made_it(cus, shared):
    # every sum of inner widths that the kernels take: workgroups of 8 to 16 wavefronts of one, two and four rows, most of which leave
    # whole wavefronts behind the last row; without a shared expert that row is a chosen expert's
    for top in (1, 2, 6):
        for width in range(64, 30720 // top + 1, 64):
            assert LIB.candy_test_unmade_choices(cus, top, width, shared) == 0, (top, width)
