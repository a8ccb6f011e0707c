"""The matrix-core line substitution (k_line_solve_m) against the one-lane
substitution: both solve the same line systems from the same factors, so on
conductive media (well-conditioned blocks) a sweep agrees to rounding.

Line lengths around what the kernel splits by: the shortest ones, odd lengths
(unequal halves), lengths that fill and miss whole groups of 2, 4 and 8
nodes, the marching right-hand sides (64 nodes and more along y and z), the
longest line of eight-line blocks (256 nodes), of two-line blocks (257 and
1024) and the first one that falls back to the one-lane kernel; one line, odd
numbers of lines and partly filled blocks.  Tolerance: 1e-11 in FP64 (a sweep
of 1024-node blocks amplifies the 1e-16 of each operation by less than 1e4 on
these media); in FP32 the stored vectors round at 6e-8 and the one-lane
kernel's line records at 6e-8 relative to corrections of the fields' own
size, 1e-5 covers both.
"""
import numpy as np
import pytest

from helpers import random_field, rel

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (2, 2, 128), (3, 2, 5), (4, 6, 3), (5, 4, 7), (6, 9, 8), (10, 12, 15), (16, 17, 14), (20, 32, 24), (33, 40, 31),
          (48, 18, 64), (63, 66, 8), (96, 7, 65), (128, 5, 96), (6, 160, 129), (4, 3, 256), (257, 4, 6), (5, 1024, 4), (4, 5, 1025)]


@pytest.mark.parametrize("precision,tol", [(0, 1e-11), (1, 1e-5)])
@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_matrix_substitution_matches_one_lane(n, precision, tol):
    from libemmi_mgfd_amd import native
    rng = np.random.default_rng(sum(n))
    xs = [np.cumsum(np.r_[0.0, rng.uniform(20.0, 60.0, m)]).astype(np.float32) for m in n]
    sig = rng.uniform(0.5, 2.0, (n[2], n[1], n[0])).astype(np.float32)
    L = native.lib()
    u, f = random_field(n, 41), random_field(n, 42)
    S = native.Solver(n, *xs, sig, sig, sig, 2 * np.pi * 100.0, precision=precision)
    prev = L.emmi_set_line_kernel(0)
    try:
        for axis in range(3):
            print(f"line sweep {n} precision {precision} axis {axis}", flush=True)
            outs = []
            for mode in (0, 1):
                L.emmi_set_line_kernel(mode)
                outs.append(S.check_op(1, 0, 0, axis, axis % 2, u, f))
            assert np.all(np.isfinite(outs[0]))
            print("  rel", rel(outs[0], outs[1]), flush=True)
            assert rel(outs[0], outs[1]) < tol
    finally:
        L.emmi_set_line_kernel(prev)
        S.close()
