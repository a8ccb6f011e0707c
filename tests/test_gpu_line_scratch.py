"""Line records in memory are allocated where a sweep can need them: a solver
whose lines have their records in LDS takes no memory for them until the
one-lane kernel is asked for, one with longer lines does from its first solve.
The batched solve of several slots is the same either way, to the order of the
sums: 1e-9 after two cycles on conductive media, where a sweep agrees to 1e-11
(3e-16 measured).
"""
import numpy as np
import pytest
import torch

from helpers import random_field, rel

pytestmark = pytest.mark.gpu


def solver(n, nslots, precision):
    from libemmi_mgfd_amd import native
    rng = np.random.default_rng(3)
    xs = [np.cumsum(np.r_[0.0, rng.uniform(20.0, 60.0, m)]).astype(np.float32) for m in n]
    sig = rng.uniform(0.5, 2.0, (n[2], n[1], n[0])).astype(np.float32)
    return native.Solver(n, *xs, sig, sig, sig, [2 * np.pi * 10.0 * (k + 1) for k in range(nslots)], precision=precision,
                         tol=1e-30, ncycle=2, graphs=0)   # (graphs take memory of their own)


@pytest.mark.parametrize("n,long_lines", [((128, 96, 80), False), ((8, 12, 1040), True)], ids=["128x96x80", "8x12x1040"])
def test_records_in_memory_on_demand(n, long_lines):
    from libemmi_mgfd_amd import native
    L = native.lib()
    ns = 3
    S = solver(n, ns, 0)
    nb = 16 * S.nvec
    b = [native.DeviceBuffer(nb).upload(random_field(n, 60 + k).reshape(-1)) for k in range(ns)]
    x, h = [native.DeviceBuffer(nb) for _ in range(ns)], [native.DeviceBuffer(nb) for _ in range(ns)]

    def solve():
        print(f"batched solve {n}", flush=True)
        S.solve_batch_device([v.ptr for v in b], [v.ptr for v in x], [v.ptr for v in h])
        return [v.download(np.complex128) for v in x]

    prev = L.emmi_set_line_kernel(0)
    try:
        matrix = solve()
        free = torch.cuda.mem_get_info()[0]
        L.emmi_set_line_kernel(1)
        one_lane = solve()
        grown = free - torch.cuda.mem_get_info()[0]
    finally:
        L.emmi_set_line_kernel(prev)
        S.close()
    for a, c in zip(matrix, one_lane):
        print("  rel", rel(a, c), flush=True)
        assert np.all(np.isfinite(a)) and rel(a, c) < 1e-9
    # of the largest colour: 80 bytes a node for a quarter of the lines (20 MB a
    # slot for 128 x 96 x 80: an allocation of its own each)
    need = ns * 80 * n[0] * n[1] * n[2] // 4
    print("  grown", grown, "records", need, flush=True)
    assert grown == 0 if long_lines else grown >= need
