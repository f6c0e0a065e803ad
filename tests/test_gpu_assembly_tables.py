"""The dense operator assembled from the meshes against the blocks of the host
Green's functions (every pair evaluated): over a mantle on a uniform
horizontal grid the assembly evaluates the pairs that differ by their
horizontal offset only and writes them out.

K_fm and K_mm agree to the rounding of the shifted coordinates, 1e-12 of the
block's largest.  Mantle spacings that miss a whole number of
fault spacings by more than the coordinates' rounding, and cells whose heights
or depths differ along a line in their last bit, keep the pair kernels: the
mismatch adds up over the columns, and a cell face through a patch centre
would move over it.  Okada's closed form (K_mf) loses digits where R + xi cancels
(1e-10 of the block against extended precision, from the patches' own
coordinates as from shifted ones), so K_mf is held to the Green's functions'
1e-10 against the oracle.  Where the rule sends a block to the pair kernels it
is equal bit for bit."""
import numpy as np
import pytest

import oetqf_amd as oq
from helpers import relerr, rs_props, visc_props

pytestmark = pytest.mark.gpu
LAM, MU = 3e10, 2e10

#        nx, nxi, dip, cells, spread (mantle x spacing / extent), x shift of the mantle, nrept, blocks from pairs
#        and, optionally, what is done to the mantle's coordinates
CASES = {
    "m=4": (16, 3, 90.0, (4, 4, 2), 1.0, 0.0, 2, ""),
    "m=1, one layer": (9, 2, 60.0, (9, 5, 1), 1.0, 0.0, 2, ""),
    "m=3, odd rows": (15, 4, 90.0, (5, 2, 3), 1.0, 0.0, 0, ""),
    "gaps between cells": (16, 3, 75.0, (4, 4, 2), 0.7, 0.0, 2, ""),
    "mantle set off": (12, 3, 90.0, (6, 4, 2), 1.0, 0.3, 1, ""),
    "spacings that do not divide": (17, 3, 90.0, (4, 4, 2), 1.0, 0.0, 2, "fm mf"),
    "one cell along x": (8, 3, 90.0, (1, 8, 2), 1.0, 0.0, 2, "fm mf"),
    "few cells": (8, 3, 90.0, (4, 1, 2), 1.0, 0.0, 2, "mf mm"),
    "cells centred on the fault plane and its patch edges": (12, 3, 90.0, (6, 3, 2), 1.0, 0.0, 2, "mf"),
    "patch centres on cell faces": (8, 3, 90.0, (4, 4, 2), 1.0, 0.25, 2, "fm"),
    "spacing off by 5e-10": (16, 3, 90.0, (4, 4, 2), 1.0, 0.0, 2, "fm mf", "stretch"),
    "spacing off by an ulp or two": (16, 3, 90.0, (4, 4, 2), 1.0, 0.0, 2, "", "stretch_ulp"),
    "one column's centres off by 1e-12 of a cell": (16, 3, 90.0, (4, 4, 2), 1.0, 0.0, 2, "fm mf mm", "column"),
    "one column's faces along y a bit off the fault plane": (16, 3, 90.0, (4, 4, 2), 1.0, 0.0, 2, "fm mf", "face"),
    "one cell's depth a bit off its layer": (16, 3, 90.0, (4, 4, 2), 1.0, 0.0, 2, "fm mf mm", "depth"),
}


def _edit(ma, how, hx):
    """The mantle's coordinates changed by less than the grid operator's own
    tolerance (1e-9 of the spacing, 1e-11 of a cell)."""
    if how in ("stretch", "stretch_ulp"):
        f = 1.0 + (5e-10 if how == "stretch" else 3e-16)
        ma.cx, ma.qx, ma.dx = ma.cx * f, ma.qx * f, ma.dx * f
    if how == "column":
        ma.cx = ma.cx.copy()
        ma.cx[1::4] += 1e-12 * hx * 8  # 8e-8 m; its faces stay
    if how == "face":  # the cells of column 2 above the fault plane y = 0 start just past it
        ma.qy = ma.qy.copy()
        c = np.nonzero(ma.qy == 0.0)[0]
        assert len(c)
        ma.qy[c[2::4]] = 1e-12
    if how == "depth":
        ma.qz = ma.qz.copy()
        ma.qz[5] = np.nextafter(ma.qz[5], 0.0)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("qtype", ["Gauss1", "Gauss2"])
def test_dense_assembly_matches_the_pair_kernels(oracle, rng, name, qtype):
    nx, nxi, dip, cells, spread, shift, nrept, pairs = CASES[name][:8]
    mf = oq.gen_mesh("RectOkada", 40e3, 12e3, 40e3 / nx, 12e3 / nxi, dip)
    ma = oq.hex8_box(-20e3, -6e3, -8e3, 40e3, 12e3, -12e3, *cells)
    hx = 40e3 / cells[0]
    ma.cx, ma.qx, ma.dx = ma.cx + shift * hx, ma.qx + shift * hx, ma.dx * spread
    if len(CASES[name]) > 8:
        _edit(ma, CASES[name][8], hx)
    pf, pa = rs_props(mf, rng), visc_props(ma, rng, 0.0)
    u = oq.ArrayPartition(np.full(pf.a.shape, pf.vpl), pf.L / pf.vpl, np.zeros((ma.ne, 6)), np.zeros((ma.ne, 6)),
                          np.zeros(pf.a.shape))
    kw = dict(ftype=oq.DipSlip(), nrept=nrept, qtype=qtype)
    p = oq.assemble_from_mesh(mf, ma, LAM, MU, pf, pa, u, (0.0, 1.0), **kw)
    K, nf = p.f.dense_operator(), mf.nx * mf.nxi
    p.f.close()
    want = dict(fm=oq.stress_greens_function(ma, mf, LAM, MU, ftype=oq.DipSlip()),
                mf=oq.stress_greens_function(mf, ma, LAM, MU, **kw),
                mm=oq.stress_greens_function(ma, LAM, MU, qtype=qtype, checkeigvals=False))
    got = dict(fm=K[:nf, nf:], mf=K[nf:, :nf], mm=K[nf:, nf:])
    if qtype == "Gauss2":  # no receiver on the fault plane or on an edge: its lines are off both
        pairs = pairs.replace("mf", "") if name.startswith(("cells centred", "few")) else pairs
    for k in got:
        if k in pairs.split():
            assert np.array_equal(got[k], want[k]), k
        elif k == "mf":
            qc, qw = oq.get_quadrature(qtype)
            ref = oracle.gf_mf(mf, ma, LAM, MU, ftype=1, qc=qc, qw=qw, nrept=nrept)
            assert relerr(got[k], ref) <= 1e-10
        else:
            assert np.abs(got[k] - want[k]).max() <= 1e-12 * np.abs(want[k]).max(), k
