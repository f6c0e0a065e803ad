"""The operators of ensembles and grouped batches, which have hex8 pair kernels
of their own (csrc/hex8_seq_dev.h) and no host entry point: K_fm and K_mm of
those kernels against the oracle at the Green's functions' 1e-10, and, column
by column, the operator that a batch really holds against the single FP64
model's, to the rounding of FP32 storage and sums (and the Green's functions'
1e-10 of a block's largest entry, for those that vanish by symmetry).  Cells near the fault,
touching the surface and in thin layers."""
import ctypes

import numpy as np
import pytest

import oetqf_amd as oq
from helpers import relerr
from oetqf_amd import _lib

pytestmark = pytest.mark.gpu
LAM, MU = 3e10, 2e10
LAUNCH = "_ZN2oq18launch_gf_hex8_seqERKNS_7DevHex8ERKNS_8DevFaultEPKdS7_iddiPdS8_lP12ihipStream_t"
BOXES = [(0.0, 20e3), (-500.0, 3e3), (-8e3, 12e3)]  # top and thickness of the mantle


class DevFault(ctypes.Structure):  # csrc/oq_internal.h
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "ax", "y", "z", "axi")] + \
               [(n, ctypes.c_int64) for n in ("nx", "nxi")] + \
               [(n, ctypes.c_double) for n in ("lrept", "dep", "sd", "cd", "s2d", "c2d")]


class DevHex8(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("cx", "cy", "cz", "qx", "qy", "qz", "dx", "dy", "dz")] + \
               [("ne", ctypes.c_int64)]


class _Device:
    def __init__(self):
        _lib.load()
        self.rt, self.bufs = ctypes.CDLL("libamdhip64.so.7"), []

    def put(self, a):
        a = np.ascontiguousarray(a, dtype=np.float64).reshape(-1)
        p = ctypes.c_void_p()
        assert self.rt.hipMalloc(ctypes.byref(p), ctypes.c_size_t(a.nbytes)) == 0
        self.bufs.append(p)
        assert self.rt.hipMemcpy(p, a.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(a.nbytes), 1) == 0
        return p

    def get(self, p, shape):
        out = np.empty(shape)
        assert self.rt.hipMemcpy(out.ctypes.data_as(ctypes.c_void_p), p, ctypes.c_size_t(out.nbytes), 2) == 0
        return out

    def close(self):
        for p in self.bufs:
            self.rt.hipFree(p)


def _meshes(top, thick, cells, dip=70.0, **kw):
    return (oq.gen_mesh("RectOkada", 40e3, 12e3, 5e3, 3e3, dip),
            oq.hex8_box(-22e3, -7e3, top, 44e3, 14e3, -thick, *cells, **kw))


@pytest.mark.parametrize("top,thick", BOXES)
@pytest.mark.parametrize("ftype,qtype", [(0, "Gauss1"), (1, "Gauss2")])
def test_batch_pair_kernels_match_the_oracle(oracle, top, thick, ftype, qtype):
    mf, ma = _meshes(top, thick, (3, 2, 2), rfx=0.5)
    qc, qw = oq.get_quadrature(qtype)
    nf, m6 = mf.nx * mf.nxi, 6 * ma.ne
    ld = m6 + 3
    launch = getattr(_lib.load(), LAUNCH)
    launch.restype = ctypes.c_int
    launch.argtypes = [ctypes.POINTER(DevHex8), ctypes.POINTER(DevFault), ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int,
                       ctypes.c_double, ctypes.c_double, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64,
                       ctypes.c_void_p]
    dev = _Device()
    try:
        f = DevFault(dev.put(mf.x), dev.put(mf.ax), dev.put(mf.y), dev.put(mf.z), dev.put(mf.axi), mf.nx, mf.nxi, 0.0,
                     mf.dep, oq.sind(mf.dip), oq.cosd(mf.dip), oq.sind(2 * mf.dip), oq.cosd(2 * mf.dip))
        h = DevHex8(*[dev.put(getattr(ma, k)) for k in ("cx", "cy", "cz", "qx", "qy", "qz", "dx", "dy", "dz")], ma.ne)
        fm, mm = dev.put(np.full((nf, ld), np.nan)), dev.put(np.full((m6, ld), np.nan))
        rc = launch(ctypes.byref(h), ctypes.byref(f), dev.put(qc), dev.put(qw), len(np.ravel(qw)), LAM, MU, ftype, fm, mm, ld,
                    None)
        assert rc == 0
        Kfm, Kmm = dev.get(fm, (nf, ld))[:, :m6], dev.get(mm, (m6, ld))[:, :m6]  # waits for the default stream
    finally:
        dev.close()
    rfm, rmm = oracle.gf_fm(ma, mf, LAM, MU, ftype=ftype, nquad=6), oracle.gf_mm(ma, LAM, MU, qc=qc, qw=qw, nquad=6)
    assert relerr(Kfm, rfm) <= 1e-10 and np.abs(Kfm - rfm).max() <= 1e-10 * np.abs(rfm).max()
    assert relerr(Kmm, rmm) <= 1e-10 and np.abs(Kmm - rmm).max() <= 1e-10 * np.abs(rmm).max()


VPL, GAMMA, STRESS, L = 2.0 ** -30, 2.0 ** -64, 2.0 ** 20, 2.0 ** -7  # sources are powers of two: exact in FP32


@pytest.mark.parametrize("top,thick", BOXES)
@pytest.mark.parametrize("kind", ["ensemble", "group"])
def test_batch_holds_the_single_models_operator(top, thick, kind):
    """Every state has one source: a patch at twice the plate rate, or one
    stress component of one cell (a diagonal one acts with its deviator)."""
    mf, ma = _meshes(top, thick, (3, 2, 2))
    shp, nf, ne = (mf.nx, mf.nxi), mf.nx * mf.nxi, ma.ne
    pf = oq.RateStateQuasiDynamicProperty(np.full(shp, 0.015), np.full(shp, 0.019), np.full(shp, L), np.full(shp, 5e7),
                                          4.9e6, VPL)
    pa = oq.PowerLawViscosityProperty(np.full(ne, GAMMA), np.zeros(ne), np.zeros(6))
    states, sources = [], []
    for j in range(nf + 6 * ne):
        v, s, src = np.full(nf, VPL), np.zeros((ne, 6)), np.zeros(nf + 6 * ne)
        if j < nf:
            v[j] = 2 * VPL
            src[j] = VPL
        else:
            c, k = (j - nf) % ne, (j - nf) // ne
            s[c, k] = 3 * STRESS if k in (0, 3, 5) else STRESS
            for q, x in ([(q, 2.0 if q == k else -1.0) for q in (0, 3, 5)] if k in (0, 3, 5) else [(k, 1.0)]):
                src[nf + q * ne + c] = x * STRESS * GAMMA
        v = v.reshape(shp, order="F")
        states.append(oq.ArrayPartition(v, L / v, np.zeros((ne, 6)), s, np.zeros(shp)))
        sources.append(src)
    S = np.array(sources)
    p = oq.assemble_from_mesh(mf, ma, LAM, MU, pf, pa, states[0], (0.0, 1.0))
    K, want = p.f.dense_operator(), []
    for u in states:
        d = oq.similar(u)
        p.f(d, u, None, 0.0)
        want.append(d)
    p.f.close()
    U, M = np.stack([u.pack() for u in states]), 16
    if kind == "ensemble":
        b = oq.Ensemble(mf, ma, LAM, MU, [pf] * len(U), pa, kdtype="fp32")
        got = b.eval(U)
    else:
        b = oq.Group([(mf, ma, pa)], LAM, MU, [[pf] * M])
        rows = []
        for i in range(0, len(U), M):
            part = np.resize(U[i:i + M], (M, U.shape[1]))
            rows.append(b.unpack(b.eval(b.pack([part])))[0][:len(U[i:i + M])])
        got = np.concatenate(rows)
    b.close()
    tau = S @ K.T  # (state, row)
    bound = 3 * 2.0 ** -24 * (np.abs(S) @ np.abs(K).T)  # an entry's rounding to FP32 and two sums
    for r in (slice(0, nf), slice(nf, None)):
        for c in (slice(0, nf), slice(nf, None)):
            bound[:, r] += 1e-10 * np.abs(K[r, c]).max() * np.abs(S[:, c]).sum(axis=1, keepdims=True)
    for i, (w, g) in enumerate(zip(want, got)):
        g = oq.similar(w).unpack(g)
        ds = np.abs(g.x[3] - w.x[3]).ravel(order="F")
        assert np.all(ds <= bound[i, nf:]), "column %d" % i
        # at steady state dv is the traction rate over the rows' impedance
        dv, wv = np.abs(g.x[0] - w.x[0]).ravel(order="F"), np.abs(w.x[0]).ravel(order="F")
        assert np.all(dv * np.abs(tau[i, :nf]) <= bound[i, :nf] * wv), "column %d" % i
