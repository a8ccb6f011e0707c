"""The matrix-core line substitution (k_line_solve_m) against the one-lane
substitution: both solve the same line systems from the same factors, so on
conductive media (well-conditioned blocks) a sweep agrees to rounding.

Line lengths around what the kernel splits by: the shortest ones, odd lengths
(unequal halves), lengths that fill and miss whole groups of 2, 4 and 8
nodes, the marching right-hand sides (64 nodes and more along y and z), the
longest line of eight-line blocks (256 nodes), of two-line blocks (257 and
1024) and lines whose records are in memory (1025 and more, or many lines of
400 nodes; runs of one node and of eight, the last block partly filled); many
lines of four nodes; one line, odd numbers of lines and partly filled blocks.  Tolerance: 1e-11 in FP64 (a sweep
of 1024-node blocks amplifies the 1e-16 of each operation by less than 1e4 on
these media); in FP32 the stored vectors round at 6e-8 and the one-lane
kernel's line records at 6e-8 relative to corrections of the fields' own
size, 1e-5 covers both.
"""
import ctypes as C

import numpy as np
import pytest

from helpers import random_field, rel

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (2, 2, 128), (3, 2, 5), (4, 6, 3), (5, 4, 7), (6, 9, 8), (10, 12, 15), (16, 17, 14), (20, 32, 24), (33, 40, 31),
          (48, 18, 64), (63, 66, 8), (96, 7, 65), (128, 5, 96), (6, 160, 129), (4, 3, 256), (257, 4, 6), (5, 1024, 4), (4, 5, 1025), (4, 130, 130), (98, 98, 400),
          (1025, 4, 3), (2, 1100, 2), (1100, 13, 7), (9, 1031, 12), (14, 7, 1026), (2, 2, 2048)]


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


@pytest.mark.parametrize("n,axis,precision,tol", [((132, 132, 258), 2, 0, 1e-10), ((132, 132, 258), 2, 1, 1e-5),
                                                  ((386, 132, 132), 0, 1, 1e-5), ((184, 130, 184), 1, 1, 1e-5)],
                         ids=["z258_fp64", "z258_fp32", "x386_fp32", "y130_fp32"])
def test_lines_of_a_colour_are_solved_exactly(n, axis, precision, tol):
    """Colours of many long lines, whose factor records lie across the lines
    (the one-lane kernel reads them, in every mode).  The sweep's last colour
    leaves no residual on the edges of its lines, up to the rounding of the
    stored vectors (6e-8 of A u in FP32; u is random, so that the residual
    before the sweep is of that size)."""
    from libemmi_mgfd_amd import native
    rng = np.random.default_rng(sum(n))
    xs = [np.cumsum(np.r_[0.0, rng.uniform(20.0, 60.0, m)]).astype(np.float32) for m in n]
    sig = rng.uniform(0.5, 2.0, (n[2], n[1], n[0])).astype(np.float32)
    u, f = random_field(n, 51), random_field(n, 52)
    S = native.Solver(n, *xs, sig, sig, sig, 2 * np.pi * 100.0, precision=precision)
    b, c = (axis + 1) % 3, (axis + 2) % 3
    for it, odd in ((0, 1), (1, 0)):   # last colour: both parities odd, both even
        nl = [len(range(1 if odd else 2, n[q], 2)) for q in (b, c)]
        assert native.lib().emmi_line_route(8 if precision == 0 else 4, axis, 1, (C.c_int * 1)(n[axis]),
                                            (C.c_long * 1)(nl[0] * nl[1])) == 0
        print(f"line sweep {n} axis {axis} precision {precision} order {it}", flush=True)
        out = S.check_op(1, 0, 0, axis, it, u, f)
        r0 = S.check_op(0, 0, 0, 0, 0, u, f).reshape(3, n[2] + 1, n[1] + 1, n[0] + 1)
        r1 = S.check_op(0, 0, 0, 0, 0, out, f).reshape(r0.shape)
        for comp in (axis, b, c):
            sel = [slice(None)] * 3   # (z, y, x) of the edges of the colour's lines
            for q in (b, c):   # component b holds the edges at pb - 1 and pb: every one along b
                sel[2 - q] = slice(1 if odd else 2, n[q], 2) if q != comp else slice(0 if odd else 1, n[q] - (n[q] + odd) % 2)
            sel[2 - axis] = slice(0, n[axis]) if comp == axis else slice(1, n[axis])
            a0, a1 = np.abs(r0[comp][tuple(sel)]).max(), np.abs(r1[comp][tuple(sel)]).max()
            print("  component", comp, a1 / a0, flush=True)
            assert a1 < tol * a0
    S.close()
