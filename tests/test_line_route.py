"""Which line substitution a launch takes (host rule, no GPU).

The matrix-core kernels size their records, LDS and node groups for one line
length, so a pack whose jobs differ in length takes the one-lane kernel, which
reads each job's own length.  Lines of up to 256 nodes have their records in
LDS; up to 1024 nodes too unless a launch has many of them; longer ones in
memory; colours of more than 4096 long lines take the one-lane kernel."""
import ctypes as C

import pytest

from libemmi_mgfd_amd import native

ONE_LANE, MATRIX, MATRIX_MEM = 0, 1, 2


def route(*cells, lines=16, esize=8, axis=1):
    n = len(cells)
    return native.lib().emmi_line_route(esize, axis, n, (C.c_int * n)(*cells), (C.c_long * n)(*[lines] * n))


@pytest.mark.parametrize("esize", [4, 8])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_equal_lengths(esize, axis):
    for n in (2, 3, 8, 31, 64, 96, 256, 257, 1024):
        assert route(n, esize=esize, axis=axis) == route(*[n] * 16, esize=esize, axis=axis) == MATRIX
    for n in (1025, 1100, 4096):
        assert route(n, esize=esize, axis=axis) == route(n, lines=4096, esize=esize, axis=axis) == MATRIX_MEM
    # the LDS holds lines of up to 256 nodes eight at a time, whatever their number
    assert route(128, lines=20000, esize=esize, axis=axis) == route(256, lines=4096, esize=esize, axis=axis) == MATRIX
    assert route(1024, lines=4096, esize=esize, axis=axis) == MATRIX_MEM
    assert route(1024, lines=4097, esize=esize, axis=axis) == route(2000, lines=9000, esize=esize, axis=axis) == ONE_LANE


@pytest.mark.parametrize("cells", [(64, 32), (8, 8, 12), (96, 96, 95), (128, 127), (2, 4), (33, 64), (1025, 1026), (300, 1100)])
def test_unequal_lengths_take_one_lane(cells):
    assert route(*cells) == ONE_LANE and route(*cells[::-1]) == ONE_LANE


def test_forced_mode_and_bad_arguments():
    L = native.lib()
    prev = L.emmi_set_line_kernel(1)
    try:
        assert route(64) == route(1100) == ONE_LANE
    finally:
        L.emmi_set_line_kernel(prev)
    assert route(*[4] * 17) == route(4, esize=2) == route(4, axis=3) == -1
