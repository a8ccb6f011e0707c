"""What is measured: the calls a program makes that models and inverts marine controlled-source surveys.

Four families, each through the package's public entry points:

* ``solve``     a solver kept per earth; a pass injects the sources, solves (one right-hand side, several frequencies of a shot, or
                several shots and frequencies in one survey solver) and extracts the receiver data;
* ``gradient``  the same solver used twice per pass: forward solves, adjoint sources from the data residuals, adjoint solves, and the
                gradient of the misfit on the model grid;
* ``call``      a whole modelling call from the model files' arrays to receiver data, nothing kept: regridding, hierarchy, factors,
                solve and release (``legacy``: the reference's own call sequence on host vectors, ``survey``: ``survey.SurveyRun``);
* ``net``       the initial-guess network: a guess for one solve, a training step, and one convolution layer forward and backward.

Earths are the package's own random marine models (``configs.config4``) and, for grids too small for their depth, ``configs.tiny``.
"""
from __future__ import annotations

import ctypes as C
import dataclasses
import io
import math
import os

import numpy as np
import torch

from libemmi_mgfd_amd import carriers, configs, native, survey, x0guess, x0net

DEV = "cuda"


# ---------------------------------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest solve: a reconnaissance grid of odd factors, complex double throughout, to the tolerance the tests use
        dict(name="solve_tiny_f64", kind="solve", n1=12, n2=10, n3=16, slots=1, shots=1, precision=0, cycleopt=2, tol=1e-8),
        # unequal axes, a V-cycle, two frequencies of one shot in FP32-storage cycles
        dict(name="solve_ragged_v", kind="solve", n1=40, n2=24, n3=36, slots=2, shots=1, precision=1, cycleopt=1, tol=1e-6),
        # plain double-precision modelling, one frequency, at the reference's default size
        dict(name="solve_64_f64", kind="solve", n1=64, n2=64, n3=64, slots=1, shots=1, precision=0, cycleopt=2, tol=1e-6),
        # the same on the large grid
        dict(name="solve_128_f64", kind="solve", n1=128, n2=128, n3=128, slots=1, shots=1, precision=0, cycleopt=2, tol=1e-6),
        # the three frequencies of a shot in one batched mixed-precision solve (the headline workload)
        dict(name="solve_128x3_mixed", kind="solve", n1=128, n2=128, n3=128, slots=3, shots=1, precision=1, cycleopt=2, tol=1e-6),
        # part of a survey: four shots on their own grids, two frequencies each, in one solver
        dict(name="survey_96x8_mixed", kind="solve", n1=96, n2=96, n3=96, slots=8, shots=4, precision=1, cycleopt=2, tol=1e-6),
        # misfit gradient of one shot at two frequencies on the inversion's grid
        dict(name="gradient_160x2", kind="gradient", n1=160, n2=160, n3=128, slots=2, shots=1, precision=1, cycleopt=2, tol=1e-6),
        # the reference's host program linked against the library: one frequency, host vectors, everything built per call
        dict(name="call_legacy_64", kind="call", api="legacy", n1=64, n2=64, n3=64, slots=1, shots=1, precision=0, cycleopt=2, tol=1e-6),
        # a small survey modelled once, as in an inversion whose model changes every iteration
        dict(name="call_survey_64x4", kind="call", api="survey", n1=64, n2=64, n3=64, slots=4, shots=2, precision=1, cycleopt=2, tol=1e-6),
        # the learned initial guess for one right-hand side on the network's own grid
        dict(name="net_guess_96", kind="net", what="guess", n1=96, n2=96, n3=96, cin=32, cout=9),
        # one optimiser step of the network's training
        dict(name="net_train_64", kind="net", what="train", n1=64, n2=64, n3=64, cin=32, cout=9),
        # one convolution of the network, forward, input gradient and weight gradient: the decoder's widest layer at full size
        dict(name="net_layer_96", kind="net", what="layer", n1=96, n2=96, n3=96, cin=48, cout=16),
    ]


def draw(rng):
    def logint(lo, hi, step):
        return max(lo, min(hi, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))

    what = rng.choice(["tiny", "solve", "solve", "batch", "survey", "gradient", "call", "guess", "train", "layer"])
    if what == "tiny":
        return dict(kind="solve", n1=2 * rng.randint(4, 8), n2=2 * rng.randint(4, 7), n3=2 * rng.randint(8, 9), slots=1, shots=1,
                    precision=rng.randint(0, 1), cycleopt=rng.randint(1, 3), tol=1e-8)
    if what in ("solve", "batch"):
        return dict(kind="solve", n1=logint(24, 128, 8), n2=logint(24, 128, 8), n3=logint(64, 128, 8),
                    slots=1 if what == "solve" else rng.randint(2, 4), shots=1,
                    precision=rng.randint(0, 1) if what == "solve" else 1, cycleopt=rng.choice([2, 2, 1]), tol=1e-6)
    if what == "survey":
        shots = rng.randint(2, 5)
        return dict(kind="solve", n1=logint(32, 96, 8), n2=logint(32, 96, 8), n3=logint(64, 96, 8), slots=shots * rng.randint(1, 2),
                    shots=shots, precision=1, cycleopt=2, tol=1e-6)
    if what == "gradient":
        return dict(kind="gradient", n1=logint(48, 128, 8), n2=logint(48, 128, 8), n3=logint(64, 128, 16), slots=rng.randint(1, 2),
                    shots=1, precision=1, cycleopt=2, tol=1e-6)
    if what == "call":
        api = rng.choice(["legacy", "survey"])
        shots = 1 if api == "legacy" else rng.randint(1, 3)
        return dict(kind="call", api=api, n1=logint(32, 80, 8), n2=logint(32, 80, 8), n3=64, shots=shots,
                    slots=1 if api == "legacy" else shots * rng.randint(1, 2), precision=0 if api == "legacy" else 1, cycleopt=2, tol=1e-6)
    if what == "layer":
        return dict(kind="net", what="layer", n1=logint(12, 112, 1), n2=logint(8, 96, 1), n3=logint(8, 96, 1),
                    cin=16 * rng.randint(1, 7), cout=16 * rng.randint(1, 4))
    most = 112 if what == "guess" else 64
    return dict(kind="net", what=what, n1=logint(32, most, 8), n2=logint(32, most, 8), n3=logint(32, most, 8), cin=32, cout=9)


# ---------------------------------------------------------------------------------------------------------------------------
# earths, sources and receivers
# ---------------------------------------------------------------------------------------------------------------------------
def _survey(case, seed):
    """A random earth with the case's multigrid size, shots and frequencies."""
    n1, n2, n3 = case["n1"], case["n2"], case["n3"]
    shots, nf = case["shots"], case["slots"] // case["shots"]
    rng = np.random.default_rng(1000003 * seed + 17)
    if n3 < 64:   # too few cells for config4's depths and padding
        s = configs.tiny(n1, n2, n3)
        k = np.exp(rng.normal(0.0, 0.3, (s.nz, 1, 1))).astype(np.float32)
        k[:5] = 1.0   # the sea keeps its resistivity
        for a in (s.rho11, s.rho22, s.rho33):
            a *= k
        s.sources = [(float(rng.uniform(-300, 300)), float(rng.uniform(-300, 300)), 450.0, float(rng.uniform(0, 90)), 5.0)]
    else:
        s = configs.config4(int(seed) % (1 << 30), 96)
        x, y, z, az, dip = s.sources[0]
        s.sources = [(x + float(v), y, z, az, dip) for v in np.linspace(0.0, 600.0, shots)]
    s.table = [(i + 1, r + 1) for i in range(shots) for r in range(len(s.receivers))]
    f = np.sort(np.exp(rng.uniform(math.log(0.2), math.log(1.5), nf)))
    return dataclasses.replace(s, n1=n1, n2=n2, n3=n3, freqs=[float(np.float32(v)) for v in f])


def _ok(rc):
    if rc:
        raise native.NativeError(native.lib().emmi_path_last_error().decode())


def _solver_kw(case):
    return dict(precision=case["precision"], cycleopt=case["cycleopt"], tol=case["tol"], ncycle=60)


def _prepare_solve(case, seed):
    s = _survey(case, seed)
    L = native.lib()
    scs = [carriers.ShotCarriers(s, k) for k in range(case["shots"])]
    grids = []
    for sc in scs:
        L.regrid_init(sc.acq, sc.emf)
        g = sc.grid()
        grids.append(tuple(sc.x_arrays()) + (g["sigma11"], g["sigma22"], g["sigma33"]))
    nf = len(s.freqs)
    n = (case["n1"], case["n2"], case["n3"])
    slots = [(k, f) for k in range(case["shots"]) for f in range(nf)]
    if case["shots"] == 1:
        solver = native.Solver(n, *grids[0], list(scs[0].omegas), **_solver_kw(case))
    else:
        solver = native.Solver.survey(n, grids, [k for k, _ in slots], [scs[k].omegas[f] for k, f in slots], **_solver_kw(case))
    nv = scs[0].nvec
    b = [torch.empty(nv, dtype=torch.complex128, device=DEV) for _ in slots]
    x = [torch.empty(nv, dtype=torch.complex128, device=DEV) for _ in slots]
    return dict(case=case, survey=s, scs=scs, slots=slots, solver=solver, b=b, x=x)


def _solve(st):
    solver, b, x = st["solver"], st["b"], st["x"]
    bp, xp = [v.data_ptr() for v in b], [v.data_ptr() for v in x]
    if len(b) == 1:
        solver.solve_device(bp[0], xp[0], bp[0])
    else:
        solver.solve_batch_device(bp, xp, bp)


def _inject(st):
    L = native.lib()
    for (k, f), b in zip(st["slots"], st["b"]):
        sc = st["scs"][k]
        _ok(L.emmi_inject_source_dev(sc.acq, sc.emf, f, b.data_ptr(), None))


def _extract(st):
    L = native.lib()
    for (k, f), b, x in zip(st["slots"], st["b"], st["x"]):
        sc = st["scs"][k]
        _ok(L.emmi_extract_emf_data_dev(sc.acq, sc.emf, f, x.data_ptr(), b.data_ptr(), None))


def _run_solve(st):
    _inject(st)
    _solve(st)
    _extract(st)
    return {"data": [sc.dcal.copy() for sc in st["scs"]], "E": list(st["x"]), "H": list(st["b"])}


def _prepare_gradient(case, seed):
    st = _prepare_solve(case, seed)
    s, sc = st["survey"], st["scs"][0]
    rng = np.random.default_rng(seed + 5)
    # observed data differ from the modelled ones by some per cent of each value
    st["misfit"] = (0.05 * (rng.standard_normal(sc.dcal.shape) + 1j * rng.standard_normal(sc.dcal.shape))).astype(np.complex64)
    nxyz = s.nx * s.ny * s.nz
    st["ef"] = [torch.empty(3 * nxyz, dtype=torch.complex64, device=DEV) for _ in st["slots"]]
    st["ea"] = [torch.empty(3 * nxyz, dtype=torch.complex64, device=DEV) for _ in st["slots"]]
    st["grad"] = torch.empty(2 * nxyz, dtype=torch.float32, device=DEV)
    st["phess"] = torch.empty(2 * nxyz, dtype=torch.float32, device=DEV)
    sc.emf.dsmute, sc.emf.drmute = 300.0, 150.0
    fwi = carriers.Fwi()
    fwi.npar, fwi.n, fwi.preco = 2, 2 * nxyz, 1
    st["idx"] = np.array([1, 2], np.int32)
    fwi.idxpar = st["idx"].ctypes.data_as(C.POINTER(C.c_int))
    st["fwi"] = fwi
    nf = len(s.freqs)
    st["tabs"] = [(C.c_void_p * nf)(*[v.data_ptr() for v in st[k]]) for k in ("ef", "ea")]
    return st


def _run_gradient(st):
    L = native.lib()
    sc = st["scs"][0]
    _inject(st)
    _solve(st)
    _extract(st)
    for f, x in enumerate(st["x"]):
        _ok(L.emmi_extract_electric_field_dev(sc.acq, sc.emf, f, x.data_ptr(), st["ef"][f].data_ptr(), None))
    # residuals relative to each value's own size (an uncertainty of some per cent)
    sc.dres[...] = st["misfit"] / np.maximum(np.abs(sc.dcal), 1e-20)
    for f, (b, x) in enumerate(zip(st["b"], st["x"])):
        _ok(L.emmi_inject_adj_source_dev(sc.acq, sc.emf, f, x.data_ptr(), b.data_ptr(), None))
    _solve(st)
    for f, x in enumerate(st["x"]):
        _ok(L.emmi_extract_electric_field_dev(sc.acq, sc.emf, f, x.data_ptr(), st["ea"][f].data_ptr(), None))
    _ok(L.emmi_build_gradient_dev(sc.acq, sc.emf, C.byref(st["fwi"]), st["tabs"][0], st["tabs"][1], st["grad"].data_ptr(),
                                  st["phess"].data_ptr(), None))
    return {"data": sc.dcal.copy(), "grad": st["grad"], "phess": st["phess"]}


def _run_call(st):
    case, s = st["case"], st["survey"]
    if case["api"] == "survey":
        run = survey.SurveyRun(s, precision=case["precision"], tol=case["tol"])
        run.run()
        return [run.results[k]["dcal"] for k in sorted(run.results)]
    L = native.lib()
    sc = carriers.ShotCarriers(s, 0)
    L.regrid_init(sc.acq, sc.emf)
    b, x = np.zeros(sc.nvec, np.complex128), np.zeros(sc.nvec, np.complex128)
    L.gmg_init(C.byref(sc.emf), 0)
    L.inject_source(sc.acq, sc.emf, b.ctypes.data, 0)
    L.gmg_apply(sc.nvec, b.ctypes.data, x.ctypes.data)
    L.extract_emf_data(sc.acq, sc.emf, x.ctypes.data, b.ctypes.data, 0)
    L.gmg_free()
    L.regrid_free(sc.emf)
    return {"data": sc.dcal.copy(), "E": x, "H": b}


# ---------------------------------------------------------------------------------------------------------------------------
# the network
# ---------------------------------------------------------------------------------------------------------------------------
class _View:
    """A block of the library's device memory for torch, which keeps this object, and so the block, alive."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"data": (int(buf.ptr), False), "shape": tuple(shape), "typestr": typestr, "version": 2, "strides": None}


def _view(buf, shape, typestr="<f4"):
    return torch.as_tensor(_View(buf, shape, typestr), device=DEV)


def _weights():
    d = np.load(os.path.join(os.path.dirname(x0net.__file__), "x0net_weights_96.npz"))
    return {k: d[k] for k in d.files if k != "train_loss"}


def _grid1d(case, seed):
    """Stretched node coordinates about the source and the earth's conductivities on the cells, in float32."""
    rng = np.random.default_rng(seed)
    g = {}
    for a, d0 in zip("123", (100.0, 100.0, 20.0)):
        n = case["n" + a]
        half = n // 2
        w = d0 * 1.06 ** (np.abs(np.arange(n) - half + 0.5) * min(1.0, 48.0 / half))
        x = np.concatenate([[0.0], np.cumsum(w)])
        x -= x[half] if a != "3" else x[n // 4]
        g["x" + a] = x.astype(np.float32)
        g["x%ss" % a] = np.append(0.5 * (x[1:] + x[:-1]), x[-1] + 0.5 * w[-1]).astype(np.float32)
        g["d%ss" % a] = np.append(w, w[-1]).astype(np.float32)
        g["d" + a] = g["d%ss" % a]
    n3 = case["n3"]
    z = g["x3s"][:n3]
    cond = np.where(z < 0, 1e-8, np.where(z < 1000, 3.2, np.exp(rng.uniform(np.log(0.2), np.log(2.0), n3))))
    s11 = torch.tensor(cond, dtype=torch.float32, device=DEV)[:, None, None].expand(n3, case["n2"], case["n1"]).contiguous()
    s33 = s11 * float(rng.uniform(0.4, 1.0))
    return g, s11, s33


def _field(case, seed, g, freq, src):
    """A diffusing dipole field on the edges, as one multigrid cycle leaves it: decays over skin depths, phases turn with distance,
    with a few per cent of roughness."""
    n1, n2, n3 = case["n1"], case["n2"], case["n3"]
    X = [torch.tensor(g["x" + a], dtype=torch.float64, device=DEV) for a in "123"]
    r = torch.sqrt((X[0][None, None, :] - src[0]) ** 2 + (X[1][None, :, None] - src[1]) ** 2 + (X[2][:, None, None] - src[2]) ** 2) + 100.0
    delta = x0guess.skin_depth(freq, configs.RHO_WATER)
    amp = torch.exp(-torch.clamp(r / delta, max=12.0)) / (r / 100.0) ** 2 * 1e-9
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    out = []
    for a in range(3):
        noise = 1.0 + 0.05 * torch.randn((n3 + 1, n2 + 1, n1 + 1), dtype=torch.float64, device=DEV, generator=gen)
        out.append(torch.polar(amp * noise / (1.0 + a), -r / delta + a))
    return torch.stack(out).reshape(-1).contiguous()


def _net_inputs(case, seed):
    g, s11, s33 = _grid1d(case, seed)
    rng = np.random.default_rng(seed + 1)
    freq, src = float(np.exp(rng.uniform(math.log(0.2), math.log(1.5)))), (float(rng.uniform(-40, 40)), float(rng.uniform(-40, 40)), 950.0)
    return g, s11, s33, freq, src, _field(case, seed, g, freq, src)


def _guesser(case, g, src):
    d = _weights()
    d["shape"] = np.array([case["n3"], case["n2"], case["n1"]])
    f = io.BytesIO()
    np.savez(f, **d)
    f.seek(0)
    return x0guess.Guesser((case["n1"], case["n2"], case["n3"]), g, src, configs.RHO_WATER, weights=f)


def _prepare_net(case, seed):
    n1, n2, n3 = case["n1"], case["n2"], case["n3"]
    nv = n1 * n2 * n3
    gen = torch.Generator(device=DEV).manual_seed(int(seed) + 3)
    st = dict(case=case, nv=nv)
    if case["what"] == "layer":
        ci, co = case["cin"], case["cout"]
        st["x"] = torch.randn((nv, ci), device=DEV, generator=gen).to(torch.bfloat16)
        st["g"] = (torch.randn((nv, co), device=DEV, generator=gen) / math.sqrt(nv)).to(torch.bfloat16)
        w = torch.randn((co, 27 * ci), device=DEV, generator=gen) * math.sqrt(2.0 / (27 * ci))
        st["w"] = w.to(torch.bfloat16).float()   # the layer's working copy is BF16: give it weights that it holds exactly
        st["bias"] = 0.1 * torch.randn(co, device=DEV, generator=gen)
        L = x0net._lib()
        st["wf"] = torch.empty((co, x0net.kpad(ci)), dtype=torch.bfloat16, device=DEV)
        st["wt"] = torch.empty((ci, x0net.kpad(co)), dtype=torch.bfloat16, device=DEV)
        torch.cuda.synchronize()
        if L.emmi_x0_prep_weights(st["w"].data_ptr(), ci, co, st["wf"].data_ptr(), st["wt"].data_ptr(), None):
            raise native.NativeError("prep_weights failed")
        st["zslab"] = max(1, n3 // 16)
        st["part"] = torch.empty(-(-n3 // st["zslab"]) * 27 * ci * co, device=DEV)
        st["y"] = torch.empty((nv, co), dtype=torch.bfloat16, device=DEV)
        st["dx"] = torch.empty((nv, ci), dtype=torch.bfloat16, device=DEV)
        st["dw"] = torch.empty((co, 27 * ci), device=DEV)
        st["db"] = torch.empty(co, device=DEV)
        return st
    g, s11, s33, freq, src, x1 = _net_inputs(case, seed)
    st.update(g=g, s11=s11, s33=s33, freq=freq, src=src, x1=x1)
    st["guesser"] = gs = _guesser(case, g, src)
    if case["what"] == "guess":
        st["x0"] = torch.empty_like(x1)
        return st
    st["net"] = gs.net
    st["feat"] = gs.features(s11.data_ptr(), s33.data_ptr(), freq, x1.data_ptr())
    # a correction like those the network learns: its own one, roughened, so that every layer receives a gradient
    st["tgt"] = 0.5 * torch.randn((nv, 9), device=DEV, generator=gen) + 0.2
    st["mask"] = torch.tensor([1.0, 4.0, 4.0] * 3, device=DEV).expand(nv, 9).contiguous()
    st["count"] = float(st["mask"].sum())
    return st


class _Ptr:
    def __init__(self, t):
        self.ptr = t.data_ptr()


def _run_net(st):
    case = st["case"]
    n1, n2, n3 = case["n1"], case["n2"], case["n3"]
    L = x0net._lib()
    if case["what"] == "layer":
        ci, co = case["cin"], case["cout"]
        p = {k: st[k].data_ptr() for k in ("x", "g", "wf", "wt", "bias", "part", "y", "dx", "dw", "db")}
        rc = L.emmi_x0_conv_fwd(p["x"], n3, n2, n1, ci, p["wf"], co, p["bias"], 0, x0net.SLOPE, None, p["y"], None, 0, None)
        rc |= L.emmi_x0_conv_fwd(p["g"], n3, n2, n1, co, p["wt"], ci, None, 3, x0net.SLOPE, None, p["dx"], None, 0, None)
        rc |= L.emmi_x0_conv_dw(p["x"], p["g"], n3, n2, n1, ci, co, p["part"], st["zslab"], p["dw"], p["db"], None)
        if rc:
            raise native.NativeError("a convolution failed")
        return {k: st[k] for k in ("y", "dx", "dw", "db")}
    if case["what"] == "guess":
        st["guesser"].guess(st["s11"].data_ptr(), st["s33"].data_ptr(), st["freq"], st["x1"].data_ptr(), st["x0"].data_ptr())
        return st["x0"]
    net = st["net"]
    net.forward(st["feat"])
    loss = net.loss_and_grad(_Ptr(st["tgt"]), _Ptr(st["mask"]), st["count"])
    net.backward()
    net.adam(lr=1e-4)
    return {"loss": loss, "y": _view(net.y, (net.nv, 9)),
            "gw": [_view(cv.gw, (cv.cout, 27 * cv.cin)) for cv in net.convs], "gb": [_view(cv.gb, (cv.cout,)) for cv in net.convs],
            "w": [_view(cv.w, (cv.cout, 27 * cv.cin)) for cv in net.convs]}


# ---------------------------------------------------------------------------------------------------------------------------
# the interface
# ---------------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "solve":
        return _prepare_solve(case, seed)
    if case["kind"] == "gradient":
        return _prepare_gradient(case, seed)
    if case["kind"] == "call":
        return dict(case=case, survey=_survey(case, seed))
    return _prepare_net(case, seed)


def run(state):
    kind = state["case"]["kind"]
    return {"solve": _run_solve, "gradient": _run_gradient, "call": _run_call, "net": _run_net}[kind](state)


def _depth(n):
    d = 0
    while n % 2 == 0 and n > 1:
        d, n = d + 1, n // 2
    return d + 1 if n > 2 else d


def _cycle_work(case):
    """Bytes and operations of one multigrid cycle: per line sweep, residual, restriction and prolongation each vector once."""
    n0 = (case["n1"], case["n2"], case["n3"])
    s, c = (16, 8) if case["precision"] == 0 else (8, 4)
    lmax = max(1, max(_depth(n) for n in n0))
    by = fl = 0.0
    for pat in range(3):
        n = n0
        for lev in range(lmax):
            ne, nc = 3.0 * (n[0] + 1) * (n[1] + 1) * (n[2] + 1), 1.0 * n[0] * n[1] * n[2]
            if lev == lmax - 1:
                visits, nxt, sweeps = lev + 1, n, 1
            else:
                nxt = tuple(v // 2 if a != pat and v % 2 == 0 and v > 2 else v for a, v in enumerate(n))
                sweeps = 2 * sum(v != w for v, w in zip(n, nxt))
                visits = lev + 1
            if case["cycleopt"] == 1:
                visits = 1
            sweep = 3 * ne * s + 3 * nc * c
            nec = 3.0 * (nxt[0] + 1) * (nxt[1] + 1) * (nxt[2] + 1)
            by += visits * (sweeps * sweep + (sweep + (ne + 2 * nec) * s + (2 * ne + nec) * s if lev < lmax - 1 else 0))
            fl += visits * (sweeps * nc * 700.0 + nc * 400.0)
            n = nxt
    return by / 3, fl / 3


def work(case):
    n = case["n1"] * case["n2"] * case["n3"]
    if case["kind"] != "net":
        # about one cycle per digit on these earths
        cycles = math.ceil(-math.log10(case["tol"])) * case["slots"] * (2 if case["kind"] == "gradient" else 1)
        by, fl = _cycle_work(case)
        return {"bytes": cycles * by, "flops": cycles * fl}
    ci, co = case["cin"], case["cout"]
    if case["what"] == "layer":
        return {"bytes": n * (2 * 2.0 * ci + 2.0 * ci + 2 * 2.0 * co + 2.0 * co), "flops": 3 * 54.0 * ci * co * n}
    # (channels in, channels out, level) of the network's convolutions
    convs = [(32, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 48, 2), (48, 48, 2), (48, 64, 3), (64, 64, 3),
             (112, 48, 2), (48, 48, 2), (80, 32, 1), (32, 32, 1), (48, 16, 0), (16, 16, 0), (16, 9, 0)]
    fl = sum(54.0 * a * b * n / 8 ** lev for a, b, lev in convs)
    by = sum(2.0 * (a + b) * n / 8 ** lev for a, b, lev in convs)
    if case["what"] == "guess":
        return {"bytes": by + n * (2 * 48.0 + 8.0), "flops": fl}
    return {"bytes": 3 * by, "flops": 3 * fl}


def tolerance(case):
    """Four times what the same code differs by with the line systems' sums in another order (the other line kernels), and for
    the network what one rounding to BF16 more or less shows (the first layers' gradients are 0.04 off their 64-bit values).  The loosest values are E in the air, where the operator all but
    leaves gradients free: 3e-10 (double) and 4e-7 (FP32-storage cycles) of the whole field; H and the receiver data agree to 1e-11."""
    if case["kind"] == "gradient":
        return {"rel": 2e-7, "max": 2e-5}
    if case["kind"] == "call" and case["api"] == "survey":
        return {"rel": 1e-9, "max": 4e-8}
    if case["kind"] != "net":
        return {"rel": 1e-9, "max": 4e-8} if case["precision"] == 0 else {"rel": 2e-6, "max": 4e-4}
    return {"guess": {"rel": 2e-3, "max": 0.05}, "train": {"rel": 0.03, "max": 0.9}, "layer": {"rel": 2e-3, "max": 0.02}}[case["what"]]


# ---------------------------------------------------------------------------------------------------------------------------
# 64-bit answers in plain torch
# ---------------------------------------------------------------------------------------------------------------------------
def _conv64(x, w, shape):
    """3x3x3 convolution, zero padding, x [V][Cin], w [Cout][27 Cin] with taps 9 dz + 3 dy + dx, as 27 products of matrices."""
    Z, Y, X = shape
    ci = x.shape[1]
    p = torch.nn.functional.pad(x.reshape(Z, Y, X, ci), (0, 0, 1, 1, 1, 1, 1, 1))
    out = 0
    for t in range(27):
        dz, dy, dx = t // 9, (t // 3) % 3, t % 3
        v = p[dz:dz + Z, dy:dy + Y, dx:dx + X].reshape(-1, ci)
        out = out + v @ w[:, t * ci:(t + 1) * ci].t()
    return out


def _unet64(feat, ws, bs, shape):
    def lrelu(v):
        return torch.where(v > 0, v, x0net.SLOPE * v)

    def dims(lev):
        return tuple(v >> lev for v in shape)

    def conv(i, v, lev, act=True):
        o = _conv64(v, ws[i], dims(lev)) + bs[i]
        return lrelu(o) if act else o

    ch, skips, v, i = (16, 32, 48, 64), [], feat, 0
    for lev in range(4):
        v = conv(i + 1, conv(i, v, lev), lev)
        i += 2
        if lev < 3:
            skips.append(v)
            Z, Y, X = dims(lev)
            v = v.reshape(Z // 2, 2, Y // 2, 2, X // 2, 2, ch[lev]).mean(dim=(1, 3, 5)).reshape(-1, ch[lev])
    for lev in (2, 1, 0):
        Z, Y, X = dims(lev)
        up = v.reshape(Z // 2, 1, Y // 2, 1, X // 2, 1, -1).expand(-1, 2, -1, 2, -1, 2, -1).reshape(Z * Y * X, -1)
        v = conv(i, torch.cat([up, skips[lev]], 1), lev)
        v = conv(i + 1, v, lev)
        i += 2
    return conv(i, v, 0, act=False)[:, :9]


def _features64(case, g, s11, s33, freq, src, x1):
    n1, n2, n3 = case["n1"], case["n2"], case["n3"]
    T = lambda a: torch.tensor(np.asarray(a), dtype=torch.float64, device=DEV)  # noqa: E731
    delta = x0guess.skin_depth(freq, configs.RHO_WATER)
    ds = [np.asarray(g["d%ss" % a], np.float64) for a in "123"]
    at = [int(np.clip(np.searchsorted(np.asarray(g["x" + a], np.float64), v) - 1, 0, case["n" + a] - 1)) for a, v in zip("123", src)]
    h = float((ds[0][at[0]] * ds[1][at[1]] * ds[2][at[2]]) ** (1.0 / 3.0))
    off = [T(g["x%ss" % a])[:case["n" + a]] - np.float32(v) for a, v in zip("123", src)]
    off = [off[0][None, None, :].expand(n3, n2, n1), off[1][None, :, None].expand(n3, n2, n1), off[2][:, None, None].expand(n3, n2, n1)]
    r = torch.sqrt(sum(o * o for o in off))
    cell = (T(ds[0])[:n1][None, None, :] * T(ds[1])[:n2][None, :, None] * T(ds[2])[:n3][:, None, None]) ** (1.0 / 3.0)
    f = [torch.log10(s11.double().clamp(min=1e-12)), torch.log10(s33.double().clamp(min=1e-12))]
    f += [(o / delta).clamp(-8, 8) for o in off]
    f += [torch.log10(r / delta + 1e-3), torch.log10(cell / delta), torch.exp(-(r / h) ** 2), torch.ones_like(r)]
    e = x1.reshape(3, n3 + 1, n2 + 1, n1 + 1)[:, :n3, :n2, :n1]
    for a in range(3):
        inside = torch.ones((n3, n2, n1), dtype=torch.bool, device=DEV)
        for ax in range(3):   # 0 = x, the last dimension
            if ax != a:
                inside.select(2 - ax, 0).fill_(False)
        v = torch.where(inside, e[a], torch.zeros_like(e[a]))
        amp = v.abs()
        big = amp > x0net.EREF
        f.append(0.1 * torch.log(amp.clamp(min=x0net.EREF) / x0net.EREF))
        f += [torch.where(big, c / amp.clamp(min=1e-300), torch.zeros_like(amp)) for c in (v.real, v.imag)]
    f += [torch.zeros_like(r)] * (32 - len(f))
    return torch.stack(f, -1).reshape(-1, 32)


def _edges64(case, y, x1):
    n1, n2, n3 = case["n1"], case["n2"], case["n3"]
    e = x1.reshape(3, n3 + 1, n2 + 1, n1 + 1)
    out = torch.zeros_like(e)
    q = y.reshape(n3, n2, n1, 9)
    for a in range(3):
        ph = torch.complex(1.0 + q[..., 3 * a + 1], q[..., 3 * a + 2])
        v = e[a, :n3, :n2, :n1] * torch.exp(q[..., 3 * a].clamp(-20, 20)) * ph / ph.abs()
        for ax in range(3):
            if ax != a:
                v.select(2 - ax, 0).fill_(0)
        out[a, :n3, :n2, :n1] = v
    return out.reshape(-1)


def _net_exact(case, seed):
    shape = (case["n3"], case["n2"], case["n1"])
    st = _prepare_net(case, seed)
    if case["what"] == "layer":
        x, g, w = st["x"].double(), st["g"].double(), st["w"].double().requires_grad_()
        x.requires_grad_()
        z = _conv64(x, w, shape)
        z.backward(g)
        y = z.detach() + st["bias"].double()
        return {"y": torch.where(y > 0, y, x0net.SLOPE * y), "dx": x.grad, "dw": w.grad, "db": g.sum(0)}
    d = _weights()
    ws = [torch.tensor(d["w%d" % i], dtype=torch.float64, device=DEV) for i in range(15)]
    bs = [torch.tensor(d["b%d" % i], dtype=torch.float64, device=DEV) for i in range(15)]
    feat = _features64(case, st["g"], st["s11"], st["s33"], st["freq"], st["src"], st["x1"])
    if case["what"] == "guess":
        return _edges64(case, _unet64(feat, ws, bs, shape), st["x1"])
    for p in ws + bs:
        p.requires_grad_()
    y = _unet64(feat, ws, bs, shape)
    # the network's loss: the mask enters its value squared and the gradient that the layers receive once
    off = (y - st["tgt"].double()).detach() * st["mask"].double()
    loss = (off ** 2).sum() / st["count"]
    y.backward(2.0 * off / st["count"])
    return {"loss": float(loss), "y": y.detach(), "gw": [w.grad for w in ws], "gb": [b.grad for b in bs], "w": [None] * 15}


def _tiny_exact(case, seed):
    """E and H of a small grid by a dense solve of the curl-curl equation, assembled here from the grid and the medium."""
    st = _prepare_solve(case, seed)
    _inject(st)
    sc = st["scs"][0]
    n = (case["n1"], case["n2"], case["n3"])
    dim = tuple(v + 1 for v in n)
    nc = dim[0] * dim[1] * dim[2]
    omu = float(sc.omegas[0]) * 4e-7 * math.pi
    X = [np.asarray(v, np.float64) for v in sc.x_arrays()]
    W = [np.append(np.diff(v), 0.0) for v in X]
    mid = [np.append(0.5 * (v[1:] + v[:-1]), v[-1] + 0.5 * (v[-1] - v[-2])) for v in X]
    D = [np.diff(m, prepend=0.0) for m in mid]
    for a in range(3):
        W[a][-1] = mid[a][-1] - X[a][-1]
        D[a][0] = mid[a][0] - X[a][0]
    g = sc.grid()
    i, j, k = np.meshgrid(*[np.arange(v) for v in dim], indexing="ij")
    p = [v.transpose(2, 1, 0).reshape(-1) for v in (i, j, k)]   # x fastest
    stride = (1, dim[0], dim[0] * dim[1])
    vol = W[2][:n[2], None, None] * W[1][None, :n[1], None] * W[0][None, None, :n[0]]
    flat = np.arange(nc)
    inner, mass = [], []
    for a in range(3):
        b, c = (a + 1) % 3, (a + 2) % 3
        ok = (p[a] < n[a]) & (p[b] >= 1) & (p[b] < n[b]) & (p[c] >= 1) & (p[c] < n[c])
        sv = g["sigma%d%d" % (a + 1, a + 1)].astype(np.float64) * vol
        m = np.zeros(nc)
        for db in (0, 1):
            for dc in (0, 1):
                q = [v[ok].copy() for v in p]
                q[b] -= db
                q[c] -= dc
                m[ok] += 0.25 * sv[q[2], q[1], q[0]]
        inner.append(ok)
        mass.append(m)
    inner, mass = np.concatenate(inner), np.concatenate(mass)
    # face curls: per face normal a, (dE_c/db - dE_b/dc), with the face's weight = dual length over area
    rows, cols, vals, wt = [], [], [], np.zeros(3 * nc)
    for a in range(3):
        b, c = (a + 1) % 3, (a + 2) % 3
        ok = (p[b] < n[b]) & (p[c] < n[c]) & (p[a] <= n[a])
        f = flat[ok]
        for comp, ax, sg in ((c, b, 1.0), (b, c, -1.0)):
            h = 1.0 / W[ax][p[ax][ok]]
            rows += [a * nc + f, a * nc + f]
            cols += [comp * nc + f + stride[ax], comp * nc + f]
            vals += [sg * h, -sg * h]
        H = 0.5 * (W[a] + np.append(0.0, W[a][:-1]))
        wt[a * nc + f] = H[p[a][ok]] * W[b][p[b][ok]] * W[c][p[c][ok]]
    K = torch.sparse_coo_tensor(np.stack([np.concatenate(rows), np.concatenate(cols)]), torch.tensor(np.concatenate(vals)),
                                (3 * nc, 3 * nc)).coalesce().to_dense().to(DEV)
    ids = torch.tensor(np.flatnonzero(inner), device=DEV)
    Kd = K[:, ids]
    A = (Kd.t() @ (torch.tensor(wt, device=DEV)[:, None] * Kd)).to(torch.complex128)
    A -= torch.diag(1j * omu * torch.tensor(mass, device=DEV)[ids])
    dual = np.concatenate([((D if a != 0 else W)[0][p[0]] * (D if a != 1 else W)[1][p[1]] * (D if a != 2 else W)[2][p[2]])
                           for a in range(3)])
    rhs = st["b"][0] * torch.tensor(dual, device=DEV)
    E = torch.zeros(3 * nc, dtype=torch.complex128, device=DEV)
    E[ids] = torch.linalg.solve(A, rhs[ids][:, None])[:, 0]
    H = torch.complex(K @ E.real, K @ E.imag) / (1j * omu)
    inside = np.tile((p[0] < n[0]) & (p[1] < n[1]) & (p[2] < n[2]), 3)
    H = torch.where(torch.tensor(inside, device=DEV), H, torch.zeros_like(H))
    return {"data": [None], "E": [E], "H": [H]}


def exact(case, seed):
    if case["kind"] == "net":
        if case["what"] == "train" and case["n1"] * case["n2"] * case["n3"] > 64 ** 3:
            return None
        return _net_exact(case, seed)
    if case["kind"] == "solve" and case["n3"] < 24 and case["slots"] == 1:
        return _tiny_exact(case, seed)
    return None
