"""Performance cases of the earthquake-cycle framework, through its public entry points.

Each case is one piece of work that a user's program repeats: a right-hand
side on device or host arrays, a stretch of a cycle with one of the device
steppers, a stretch of an ensemble or of a grouped batch, Green's functions
handed to the host, and a whole model assembled from its meshes.  Sizes are
those of the workloads in oetqf_amd.workloads and bench.py, with odd and
ragged ones beside them.

The library and torch share one HIP runtime when torch is imported first, so
device states are torch tensors handed to the C ABI by address.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oetqf.jl_amd"))
import oetqf_amd as oq  # noqa: E402
from oetqf_amd import _lib, workloads  # noqa: E402

LAM = MU = 30e9  # nu = 0.25
YEAR = workloads.YEAR
ELEM = {"fp64": 8, "fp32": 4, "bf16": 2, "fp16x2": 4}
DMA_SHAPE = "dma-r64-k64-2wg"  # the tile shape the autotuner keeps for the grouped batch

BASE = dict(nx=32, nxi=16, mx=0, my=0, mz=0, kdtype="fp64", dip=90.0, grading=1.05, bump=1.0)


def _c(path, name=None, **kw):
    c = dict(BASE, path=path, **kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the reference's own contract, ode(du, u, p, t) on host arrays, on its
        # CPU-runnable fault of 512 patches with dilatancy: the smallest call,
        # what a host integrator makes twice or six times per step
        _c("rhs_host", "host rhs 512 dilatancy", grading=1.0, dila=True),
        # the fault-only right-hand side on a resident state, K_ff by DFT as
        # the reference applies it: 256 x 64 patches, the largest fault
        _c("rhs", "rhs fault 256x64 dft", nx=256, nxi=64, kdtype="fft"),
        # the headline: the composite model (4096 patches + 2048 cells) with the
        # dense FP64 operator
        _c("rhs", "rhs composite fp64", nx=128, nxi=32, mx=16, my=16, mz=8),
        # an odd-sized coupled model on a refined mantle, FP32 operator
        _c("rhs", "rhs odd coupled fp32", nx=97, nxi=21, mx=11, my=9, mz=5, kdtype="fp32", bump=0.5),
        # the composite model with every block in its translation-invariant form
        _c("rhs", "rhs composite grid", nx=128, nxi=32, mx=16, my=16, mz=8, kdtype="fft_grid"),
        # a stretch of the 512-patch cycle, Tsit5 in the persistent stepper with
        # the recorder on, as run_cycle drives it
        _c("cycle", "cycle 512 tsit5", grading=1.0, alg="tsit5", steps=512),
        # a stretch of the composite cycle, VCABM5 (the example's solver) over
        # the grid operator in the graph stepper
        _c("cycle", "cycle composite vcabm5", nx=128, nxi=32, mx=16, my=16, mz=8, kdtype="fft_grid", alg="vcabm5",
           steps=512),
        # 256 frictional realizations of the composite model, split-FP16
        # operator: a run of 48 lockstep Tsit5 steps between two looks at the states
        _c("ensemble", "ensemble 256 fp16x2", nx=128, nxi=32, mx=16, my=16, mz=8, kdtype="fp16x2", members=256,
           alg="tsit5", steps=48),
        # a small study: 24 realizations of an odd-sized model, FP32, VCABM5
        _c("ensemble", "ensemble 24 odd fp32", nx=61, nxi=17, mx=9, my=7, mz=5, kdtype="fp32", members=24,
           alg="vcabm5", steps=64),
        # 24 geometries of 1024-8192 patches (half with mantles) x 16 realizations
        _c("group", "group 24x16", geoms=24, members=16, pmin=1024, pmax=8192, alg="tsit5", steps=16),
        # the four Green's functions handed to the host, the call sequence of the
        # reference's example: a dipping fault over a mantle refined toward its
        # sides, 8-point quadrature
        _c("greens", "greens dipping refined", nx=40, nxi=20, mx=12, my=9, mz=3, dip=60.0, bump=0.5, qtype="Gauss2"),
        # the composite model assembled from its meshes and one right-hand side
        _c("assembly", "assemble composite fp64", nx=128, nxi=32, mx=16, my=16, mz=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: any path, sizes over their logarithm."""
    path = rng.choice(["rhs", "rhs", "rhs", "rhs_host", "cycle", "ensemble", "group", "greens", "assembly"])
    coupled = dict(mx=_log(rng, 4, 16), my=_log(rng, 4, 16), mz=rng.randint(2, 8))
    fault = dict(nx=_log(rng, 16, 256), nxi=_log(rng, 6, 64))
    both = dict(nx=_log(rng, 24, 128), nxi=_log(rng, 8, 32), **coupled)
    shape = dict(dip=rng.choice([90.0, 90.0, 60.0]), grading=rng.choice([1.0, 1.05]))
    bump = dict(bump=rng.choice([1.0, 0.5]))
    if path == "rhs":
        kd = rng.choice(["fp64", "fp32", "bf16", "toeplitz", "fft", "fft", "fft_grid", "fft_grid"])
        if kd == "toeplitz":
            return _c(path, kdtype=kd, **fault, **shape)
        if kd == "fft_grid":
            if rng.random() < 0.7:  # mantle spacing a multiple of the fault's
                both["nx"] = both["mx"] * max(1, min(8, round(both["nx"] / both["mx"])))
            return _c(path, kdtype=kd, **both, **shape)
        if rng.random() < 0.4:
            return _c(path, kdtype=kd, **fault, **shape)
        return _c(path, kdtype=kd, **both, **shape, **bump)
    if path == "rhs_host":
        if rng.random() < 0.5:
            return _c(path, kdtype=rng.choice(["fp64", "toeplitz", "fft"]), dila=rng.random() < 0.5, **fault, **shape)
        return _c(path, kdtype=rng.choice(["fp64", "fp32"]), **both, **shape, **bump)
    if path == "cycle":
        alg = dict(alg=rng.choice(["tsit5", "vcabm5"]), steps=_log(rng, 128, 512))
        if rng.random() < 0.5:  # small faults: the persistent stepper's range and beyond
            return _c(path, kdtype="fp64", nx=_log(rng, 16, 64), nxi=_log(rng, 6, 24), grading=shape["grading"], **alg)
        if rng.random() < 0.5:
            return _c(path, kdtype="fft", **fault, **shape, **alg)
        both["nx"] = both["mx"] * max(1, min(8, round(both["nx"] / both["mx"])))
        return _c(path, kdtype=rng.choice(["fp64", "fft_grid"]), **both, **shape, **alg)
    if path == "ensemble":
        m = dict(members=_log(rng, 5, 256), alg=rng.choice(["tsit5", "vcabm5"]), steps=_log(rng, 16, 48),
                 kdtype=rng.choice(["fp32", "fp16x2", "fp16x2", "bf16"]))
        if rng.random() < 0.3:
            return _c(path, nx=_log(rng, 24, 128), nxi=_log(rng, 8, 32), **shape, **m)
        return _c(path, **both, **shape, **bump, **m)
    if path == "group":
        lo = _log(rng, 256, 1024)
        return _c(path, geoms=rng.randint(4, 24), members=rng.randint(3, 16), pmin=lo, pmax=_log(rng, 2 * lo, 8192),
                  alg=rng.choice(["tsit5", "vcabm5"]), steps=_log(rng, 8, 16))
    if path == "greens":
        return _c(path, nx=_log(rng, 16, 64), nxi=_log(rng, 6, 24), mx=_log(rng, 4, 12), my=_log(rng, 4, 10),
                  mz=rng.randint(2, 4), qtype=rng.choice(["Gauss1", "Gauss2"]), **shape, **bump)
    return _c(path, kdtype=rng.choice(["fp64", "fp32", "fft"]), **both, **shape, **bump)


# ---------------- inputs ----------------

def _geometry(case, seed):
    """Fault of about 80 x 20 km and a mantle block below 10 km spanning it
    (cells refined toward its sides when bump < 1); the seed scales both."""
    rng = np.random.default_rng([20261202, seed])
    g = rng.uniform(0.9, 1.1)
    mf = oq.mesh.gen_mesh_graded(80e3 * g, 20e3 * g, 80e3 * g / case["nx"], case["nxi"], case["dip"],
                                 ratio=case["grading"])
    ma = None
    if case["mx"] > 0:
        ma = oq.hex8_box(-40e3 * g, -20e3 * g, -10e3 * g, 80e3 * g, 40e3 * g, -30e3 * g, case["mx"], case["my"],
                         case["mz"], rfx=case["bump"], rfy=case["bump"])
    return mf, ma, rng


def _friction(mf, ma):
    shp = (mf.nx, mf.nxi)
    d = np.broadcast_to(-mf.z, shp)
    b = workloads._b_profile(d) if ma is None else workloads._b_profile(d, bottom=8e3)
    return oq.RateStateQuasiDynamicProperty(np.full(shp, 0.015), b, np.full(shp, 0.012), np.full(shp, 50e6),
                                            MU / (2 * 3040.0), 1e-9, 0.6, 1e-6)


def _model(case, seed, spread):
    """Meshes, properties and a state: slip rates spread about the plate rate,
    states near their steady values, deviatoric stresses of about 1 MPa."""
    mf, ma, rng = _geometry(case, seed)
    pf = _friction(mf, ma)
    shp = (mf.nx, mf.nxi)
    v = pf.vpl * np.exp(spread * rng.standard_normal(shp))
    parts = [v, pf.L / v]
    pa = dila = None
    if ma is not None:
        pa = oq.PowerLawViscosityProperty(np.full(ma.ne, 1.0 / (2 * 1e19)), np.zeros(ma.ne), np.zeros(6))
        parts += [np.zeros((ma.ne, 6)), 1e6 * rng.standard_normal((ma.ne, 6))]
    parts.append(np.zeros(shp))
    if case.get("dila"):
        dila = oq.DilatancyProperty(10 ** rng.uniform(5, 7, shp), 10 ** rng.uniform(-5, -3, shp),
                                    10 ** rng.uniform(-10, -9, shp), rng.uniform(1e6, 5e6, shp))
        parts.append(dila.p0 * (1 + 0.1 * rng.standard_normal(shp)))
    return mf, ma, pf, pa, dila, oq.ArrayPartition(*parts)


def _ftype(case):
    return oq.StrikeSlip() if case["dip"] == 90.0 else oq.DipSlip()


def _problem(case, m, tspan):
    mf, ma, pf, pa, dila, u = m
    return oq.assemble_from_mesh(mf, ma, LAM, MU, pf, pa, u, tspan, ftype=_ftype(case), kdtype=case["kdtype"],
                                 dila=dila)


def _alg(case):
    return oq.Tsit5() if case["alg"] == "tsit5" else oq.VCABM5()


def _group_workloads(case, seed):
    ws = workloads.grouped_batch(G=case["geoms"], M=case["members"], pmin=case["pmin"], pmax=case["pmax"])
    rng = np.random.default_rng([20261204, seed])
    for w in ws:  # the geometries are the batch's, the initial slip rates the seed's
        nf = w["mf"].nx * w["mf"].nxi
        f = np.exp(0.1 * rng.standard_normal((case["members"], nf)))
        w["U0"][:, :nf] *= f
        w["U0"][:, nf:2 * nf] /= f
    return ws


def prepare(case, seed):
    path = case["path"]
    if path == "group":
        ws = _group_workloads(case, seed)
        grp = oq.Group([(w["mf"], w["ma"], w["pa"]) for w in ws], LAM, MU, [w["members"] for w in ws])
        grp.set_shapes({b: DMA_SHAPE for b in range(8)})
        return dict(case=case, batch=grp, U0=grp.pack([w["U0"] for w in ws]))
    if path == "ensemble":
        mf, ma, pf, pa, _, u = _model(case, seed, 0.1)
        members, U0 = workloads.ensemble_members(dict(pf=pf, ma=ma), case["members"], seed=20261203 + seed)
        ens = oq.Ensemble(mf, ma, LAM, MU, members, pa, ftype=_ftype(case), kdtype=case["kdtype"])
        return dict(case=case, batch=ens, U0=U0)
    m = _model(case, seed, 0.1 if path == "cycle" else 0.5)
    if path in ("greens", "assembly"):
        return dict(case=case, model=m)
    prob = _problem(case, m, (0.0, 300 * YEAR))
    u = m[-1]
    if path == "rhs":
        ud = torch.from_numpy(u.pack()).cuda()
        du = torch.zeros_like(ud)
        outs, o = [], 0
        for a in u.x:
            outs.append(du[o:o + a.size])
            o += a.size
        return dict(case=case, prob=prob, call=_lib.load().oq_rhs_eval_device, h=prob.f.h,
                    u=ud, du=du, up=ctypes.c_void_p(ud.data_ptr()), dup=ctypes.c_void_p(du.data_ptr()), outs=outs)
    return dict(case=case, prob=prob, u=u, du=oq.similar(u))


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "rhs":
        rc = state["call"](state["h"], 0.0, state["up"], state["dup"])
        if rc:
            _lib.check(rc)
        return state["outs"]
    if path == "rhs_host":
        state["prob"].f(state["du"], state["u"], None, 0.0)
        return [np.array(a) for a in state["du"].x]
    if path == "cycle":
        it = oq.Integrator(state["prob"], reltol=1e-6, abstol=1e-8, alg=_alg(case))
        it.record(stride=1, snap_capacity=0, step_capacity=case["steps"])
        try:
            it.set_persistent(True)
        except ValueError:
            pass  # not a small fault-only problem: the graph stepper
        it.step(case["steps"])
        st, sv, _, _ = it.drain()
        t, dt, u, na, nr = it.state()
        it.close()
        # one entry per attempted step: rejected ones leave the tail at zero
        rec = np.zeros((2, case["steps"]))
        rec[0, :len(st)] = st
        rec[1, :len(sv)] = sv
        return dict(t=t, u=list(u.x), record=rec)
    if path in ("ensemble", "group"):
        b = state["batch"]
        b.start(state["U0"], (0.0, 300 * YEAR), reltol=1e-6, abstol=1e-8, dt0=1.0, alg=_alg(case))
        b.run(case["steps"])
        t, U, na, nr, rc = b.state()
        return dict(t=t, U=U)
    mf, ma, pf, pa, dila, u = state["model"]
    if path == "greens":
        ft = _ftype(case)
        return [oq.stress_greens_function(mf, LAM, MU, ftype=ft),
                oq.stress_greens_function(mf, ma, LAM, MU, ftype=ft, qtype=case["qtype"]),
                oq.stress_greens_function(ma, mf, LAM, MU, ftype=ft),
                oq.stress_greens_function(ma, LAM, MU, qtype=case["qtype"], checkeigvals=False)]
    prob = _problem(case, state["model"], (0.0, 300 * YEAR))
    du = oq.similar(u)
    prob.f(du, u, None, 0.0)
    prob.f.close()
    return list(du.x)


# ---------------- what a pass cannot do without ----------------

def _sizes(case):
    nf, ne = case["nx"] * case["nxi"], case["mx"] * case["my"] * case["mz"]
    return nf, ne, nf + 6 * ne


def _grid_tables(case):
    """Entries of the translation-invariant blocks: K_ff by offset, K_mm by
    offset, K_fm and K_mf by offset along strike where the spacings allow it."""
    nf, ne, _ = _sizes(case)
    nx, nxi, mx, my, mz = (case[k] for k in ("nx", "nxi", "mx", "my", "mz"))
    ff = nx * nxi * nxi
    if ne == 0:
        return ff
    mm = 36 * mz * mz * (2 * mx - 1) * (2 * my - 1)
    fm = 2 * nxi * 6 * my * mz * (nx + nx // mx * (mx - 1)) if nx % mx == 0 else 2 * nf * 6 * ne
    return ff + mm + fm


def _rhs_work(case, members=1):
    nf, ne, n = _sizes(case)
    state = 8 * members * (2 * nf + 6 * ne + 3 * nf + 12 * ne + 4 * nf) + 16 * ne
    kd = case["kdtype"]
    if kd in ("fft", "toeplitz", "fft_grid"):
        entries = _grid_tables(case) if kd == "fft_grid" else case["nx"] * case["nxi"] ** 2 + 6 * ne * (n + nf)
        return dict(bytes=8 * entries + state, flops=2 * entries)  # every entry used at least once
    return dict(bytes=ELEM[kd] * n * n + state, flops=2 * n * n * members)


# multiply-adds counted per source-receiver pair: an Okada evaluation, a
# hex8 traction (K_fm) and a hex8 stress (K_mm)
DC3D, HEX_T, HEX_S = 4.3e3, 1.42e5, 2.15e5


def _greens_work(case, nq):
    """Pairs that differ: all of them on refined or incommensurate meshes."""
    nf, ne, n = _sizes(case)
    nx, nxi, mx, my, mz = (case[k] for k in ("nx", "nxi", "mx", "my", "mz"))
    flops = 5 * DC3D * nx * nxi * nxi
    if ne:
        even = case["bump"] == 1.0
        fm = nxi * my * mz * (nx + nx // mx * (mx - 1)) if even and nx % mx == 0 else nf * ne
        mm = mz * mz * (2 * mx - 1) * (2 * my - 1) if even else ne * ne
        flops += fm * (5 * nq * DC3D + HEX_T) + mm * nq * HEX_S
    return flops


def work(case):
    path = case["path"]
    if path == "group":
        ws = workloads.grouped_batch(G=case["geoms"], M=1, pmin=case["pmin"], pmax=case["pmax"])
        per = 6 if case["alg"] == "tsit5" else 2
        b = f = 0
        for w in ws:
            nf, ne = w["mf"].nx * w["mf"].nxi, (w["ma"].ne if w["ma"] is not None else 0)
            n = nf + 6 * ne
            b += 4 * n * n + 8 * case["members"] * (9 * nf + 18 * ne)
            f += 2 * n * n * case["members"]
        return dict(bytes=b * per * case["steps"], flops=f * per * case["steps"])
    if path in ("cycle", "ensemble"):
        per = (6 if case["alg"] == "tsit5" else 2) * case["steps"]
        w = _rhs_work(case, case.get("members", 1))
        return dict(bytes=w["bytes"] * per, flops=w["flops"] * per)
    nf, ne, n = _sizes(case)
    if path == "greens":
        nq = 8 if case["qtype"] == "Gauss2" else 1
        out = 16 * case["nx"] * case["nxi"] ** 2 + 8 * 12 * ne * nf + 8 * 36 * ne * ne
        return dict(bytes=out, flops=_greens_work(case, nq))
    w = _rhs_work(case)
    if path == "assembly":
        return dict(bytes=2 * w["bytes"], flops=w["flops"] + _greens_work(case, 1))
    return w


# ---------------- 64-bit values where plain numpy has them ----------------

def exact(case, seed):
    """The components of a right-hand side that involve no Green's function
    (the others' operators have no form in plain numpy that ends in seconds)."""
    if case["path"] not in ("rhs", "rhs_host", "assembly"):
        return None
    mf, ma, pf, pa, dila, u = _model(case, seed, 0.5)
    v, th = u.x[0], u.x[1]
    dth = 1.0 - v * th / pf.L
    out = [None, dth]
    if ma is not None:
        s = u.x[3]
        m = (s[:, 0] + s[:, 3] + s[:, 5]) / 3.0
        dev = s.copy()
        for k in (0, 3, 5):
            dev[:, k] -= m
        out += [np.asfortranarray(pa.γ[:, None] * dev), None]
    out.append(v.copy())
    if dila is not None:
        out.append(-(u.x[3] - dila.p0) / dila.tp + dila.eps / dila.beta / th * dth)
    if case["path"] == "rhs":
        return [None if a is None else a.reshape(-1, order="F") for a in out]
    return out
