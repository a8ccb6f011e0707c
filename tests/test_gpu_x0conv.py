"""The network's convolutions against 64-bit sums of the same BF16 values, at the
sizes where their kernels split: the forward kernel that marches through LDS
(rows of 32 voxels and more, planes of eight rows and more) with the weights in
LDS and, for many channels, in memory, with four rows instead of eight, and the
one that gathers from memory (narrower grids, 128 channels); partial tiles along
every axis, single planes and rows; the weight gradient with one, two and three
input tiles per block, groups that the channels do not fill, chunks across row
and plane ends, a slab shorter than the others, and blocks of four, eight and
sixteen waves (slabs of up to 64, up to 1024 and of more voxels).

Tolerances: products of BF16 values are exact in FP32 and sums of K = 27 Cin
terms (or of all voxels, for the weight gradient) round at 2^-24 each, so 1e-5
of the result's norm for FP32 outputs (K <= 3456); BF16 outputs round at 2^-9 =
2e-3 on top.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 32), (3, 9, 33), (3, 17, 33), (2, 16, 40), (5, 8, 64), (4, 11, 95), (1, 13, 47), (6, 7, 32), (5, 9, 31), (2, 1, 40), (3, 2, 5), (1, 1, 1)]
CHANNELS = [(16, 16), (32, 48), (48, 16), (64, 64), (80, 32), (112, 48), (128, 16), (16, 128)]


def rel(a, b):
    return float((a - b).norm() / max(float(b.norm()), 1e-30))


def taps64(x, shape):
    """[V][27][C] of x [V][C] in float64, zero outside the grid"""
    Z, Y, X = shape
    p = torch.nn.functional.pad(x.double().reshape(Z, Y, X, -1), (0, 0, 1, 1, 1, 1, 1, 1))
    return torch.stack([p[dz:dz + Z, dy:dy + Y, dx:dx + X].reshape(Z * Y * X, -1)
                        for dz in range(3) for dy in range(3) for dx in range(3)], 1)


@pytest.mark.parametrize("ci,co", CHANNELS)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_convolution_matches_64_bit(shape, ci, co):
    from libemmi_mgfd_amd import x0net
    Z, Y, X = shape
    nv = Z * Y * X
    gen = torch.Generator().manual_seed(nv + 7 * ci + co)
    x = torch.randn((nv, ci), generator=gen).to(torch.bfloat16)
    g = torch.randn((nv, co), generator=gen).to(torch.bfloat16)
    act = torch.randn((nv, co), generator=gen).to(torch.bfloat16)
    w = (torch.randn((co, 27 * ci), generator=gen) / np.sqrt(27 * ci)).to(torch.bfloat16).float()
    bias = torch.randn(co, generator=gen)
    L = x0net._lib()
    d = {k: v.cuda() for k, v in dict(x=x, g=g, act=act, w=w, bias=bias).items()}
    wf = torch.empty((co, x0net.kpad(ci)), dtype=torch.bfloat16, device="cuda")
    wt = torch.empty((ci, x0net.kpad(co)), dtype=torch.bfloat16, device="cuda")
    assert L.emmi_x0_prep_weights(d["w"].data_ptr(), ci, co, wf.data_ptr(), wt.data_ptr(), None) == 0
    t = taps64(x, shape)
    z = t.reshape(nv, -1) @ w.double().t()
    for epi in range(4):
        print(f"conv {shape} {ci}->{co} epilogue {epi}", flush=True)
        store = co - 7 if epi == 1 else 0
        ob = torch.full((nv, co), float("nan"), dtype=torch.bfloat16, device="cuda")
        of = torch.full((nv, max(store, 1)), float("nan"), device="cuda")
        rc = L.emmi_x0_conv_fwd(d["x"].data_ptr(), Z, Y, X, ci, wf.data_ptr(), co, d["bias"].data_ptr(), epi, x0net.SLOPE,
                                d["act"].data_ptr(), ob.data_ptr(), of.data_ptr(), store, None)
        assert rc == 0
        torch.cuda.synchronize()
        if epi == 0:
            r = z + bias.double()
            r = torch.where(r > 0, r, x0net.SLOPE * r)
        elif epi == 1:
            r = (z + bias.double())[:, :store]
        elif epi == 2:
            r = torch.where(act.double() > 0, z, x0net.SLOPE * z)
        else:
            r = z
        out = of.cpu().double() if epi == 1 else ob.cpu().double()
        assert rel(out, r) < (1e-5 if epi == 1 else 3e-3)
    for zslab in {1, 2, max(1, Z)}:
        print(f"weight gradient {shape} {ci}->{co} slab {zslab}", flush=True)
        part = torch.empty(-(-Z // zslab) * 27 * ci * co, device="cuda")
        dw = torch.full((co, 27 * ci), float("nan"), device="cuda")
        db = torch.full((co,), float("nan"), device="cuda")
        assert L.emmi_x0_conv_dw(d["x"].data_ptr(), d["g"].data_ptr(), Z, Y, X, ci, co, part.data_ptr(), zslab,
                                 dw.data_ptr(), db.data_ptr(), None) == 0
        torch.cuda.synchronize()
        ref = (g.double().t() @ t.reshape(nv, -1))
        assert rel(dw.cpu().double(), ref) < 1e-5 and rel(db.cpu().double(), g.double().sum(0)) < 1e-5


@pytest.mark.parametrize("shape", [(2, 9, 33), (2, 5, 7)], ids=["rows_of_33", "rows_of_7"])
def test_outputs_at_any_element_offset(shape):
    """bias, act and the outputs may start at any element of a buffer: the
    results are those of aligned ones, bit for bit, and nothing beside them is
    written."""
    from libemmi_mgfd_amd import x0net
    Z, Y, X = shape
    nv, ci, co = Z * Y * X, 16, 32
    gen = torch.Generator().manual_seed(3)
    x = torch.randn((nv, ci), generator=gen).to(torch.bfloat16).cuda()
    act = torch.randn(nv * co + 1, generator=gen).to(torch.bfloat16).cuda()
    w = torch.randn((co, 27 * ci), generator=gen).cuda()
    bias = torch.randn(co + 1, generator=gen).cuda()
    L = x0net._lib()
    wf = torch.empty((co, x0net.kpad(ci)), dtype=torch.bfloat16, device="cuda")
    wt = torch.empty((ci, x0net.kpad(co)), dtype=torch.bfloat16, device="cuda")
    assert L.emmi_x0_prep_weights(w.data_ptr(), ci, co, wf.data_ptr(), wt.data_ptr(), None) == 0
    ab, bb = act[1:].clone(), bias[1:].clone()
    for epi in (0, 2, 3):
        print(f"conv {shape} epilogue {epi}, outputs one element on", flush=True)
        outs = []
        for a, b, off in ((ab.data_ptr(), bb.data_ptr(), 0), (act.data_ptr() + 2, bias.data_ptr() + 4, 1)):
            ob = torch.full((nv * co + 2,), 7.0, dtype=torch.bfloat16, device="cuda")
            assert L.emmi_x0_conv_fwd(x.data_ptr(), Z, Y, X, ci, wf.data_ptr(), co, b, epi, x0net.SLOPE, a,
                                      ob.data_ptr() + 2 * off, None, 0, None) == 0
            torch.cuda.synchronize()
            assert float(ob[nv * co + off]) == 7.0 and (off == 0 or float(ob[0]) == 7.0)
            outs.append(ob[off:off + nv * co].clone())
        assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("shape,ci,co", [((600, 16, 64), 16, 16), ((600, 16, 64), 48, 16), ((300, 20, 45), 16, 48),
                                         ((600, 16, 64), 96, 32), ((80, 80, 80), 64, 64), ((40, 39, 41), 48, 48)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_planes_of_a_march_equal_those_of_a_slab(shape, ci, co):
    """Blocks that march through several planes (the ring of three planes in LDS
    turns more than once) against slabs of the same input, one plane per block
    or the gathering kernel: the same sums in the same order, bit for bit."""
    from libemmi_mgfd_amd import x0net
    Z, Y, X = shape
    pl = Y * X
    L = x0net._lib()
    assert L.emmi_x0_conv_route(Z, Y, X, ci, co) > 0
    gen = torch.Generator(device="cuda").manual_seed(ci + co)
    x = torch.randn((Z * pl, ci), generator=gen, device="cuda").to(torch.bfloat16)
    w = torch.randn((co, 27 * ci), generator=gen, device="cuda") / np.sqrt(27 * ci)
    bias = torch.randn(co, generator=gen, device="cuda")
    wf = torch.empty((co, x0net.kpad(ci)), dtype=torch.bfloat16, device="cuda")
    wt = torch.empty((ci, x0net.kpad(co)), dtype=torch.bfloat16, device="cuda")
    assert L.emmi_x0_prep_weights(w.data_ptr(), ci, co, wf.data_ptr(), wt.data_ptr(), None) == 0

    def conv(z0, nz):
        out = torch.full((nz * pl, co), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert L.emmi_x0_conv_fwd(x.data_ptr() + 2 * ci * z0 * pl, nz, Y, X, ci, wf.data_ptr(), co, bias.data_ptr(), 0,
                                  x0net.SLOPE, None, out.data_ptr(), None, 0, None) == 0
        torch.cuda.synchronize()
        return out.reshape(nz, pl, co)

    print(f"conv {shape} {ci}->{co}", flush=True)
    whole, n = conv(0, Z), 6
    assert bool(torch.isfinite(whole).all())
    for z0 in [*range(0, Z - n, 4), Z - n]:
        part = conv(z0, n)
        lo, hi = (0 if z0 == 0 else 1), (n if z0 == Z - n else n - 1)
        assert torch.equal(whole[z0 + lo:z0 + hi], part[lo:hi]), z0
