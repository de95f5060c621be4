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


def taken(experts, top, ff, shared, d):
    return LIB.candy_test_expert_spec(experts, top, ff, shared, d)


def test_which_specs_are_taken():
    # 64 KB for a row in f32 with a score an expert and the choice behind it
    for d in (64, 2048, 16256, 16257, 16320):
        room = 16384 - (d + 63) // 64 * 64
        for top in (1, 2, 12, 30):
            for experts in {top, 32, room - 2 * top - 1, room - 2 * top, room - 2 * top + 1}:
                if top <= experts <= 512:
                    assert taken(experts, top, 8, 0, d) == (experts + 2 * top <= room), (experts, top, d)
    assert not taken(1, 1, 8, 0, 16321)
    # 64 KB for the inner activations in bfloat16 with twelve bytes for 64 of them
    assert taken(8, 1, 29952, 0, 64) == 1 and not taken(8, 1, 29953, 0, 64)
    assert taken(8, 6, 4096, 5376, 64) == 1 and not taken(8, 6, 4096, 5377, 64)
    assert not taken(8, 8, 1 << 20, 1 << 20, 64)
