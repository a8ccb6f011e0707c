"""Which line substitution a launch takes (host rule, no GPU): the matrix-core
kernel sizes its records, LDS and node groups for one line length, so a pack
whose jobs differ in length takes the one-lane kernel, which reads each job's
own length.  Lengths of one, equal and unequal node groups (2, 4, 8)."""
import ctypes as C

import pytest

from libemmi_mgfd_amd import native

ONE_LANE, MATRIX = 0, 1


def route(*cells):
    return native.lib().emmi_line_route(len(cells), (C.c_int * len(cells))(*cells))


@pytest.mark.parametrize("n", [2, 3, 8, 31, 64, 96, 256, 257, 1024])
def test_equal_lengths_take_the_matrix_cores(n):
    assert route(n) == route(*[n] * 16) == MATRIX


@pytest.mark.parametrize("cells", [(64, 32), (8, 8, 12), (96, 96, 95), (128, 127), (2, 4), (33, 64)])
def test_unequal_lengths_take_one_lane(cells):
    assert route(*cells) == ONE_LANE and route(*cells[::-1]) == ONE_LANE


def test_forced_mode_and_bad_counts():
    L = native.lib()
    prev = L.emmi_set_line_kernel(1)
    try:
        assert route(64) == ONE_LANE
    finally:
        L.emmi_set_line_kernel(prev)
    assert L.emmi_line_route(0, (C.c_int * 1)(4)) == -1 and L.emmi_line_route(17, (C.c_int * 17)(*[4] * 17)) == -1
