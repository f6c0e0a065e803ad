"""The grid operator against the dense operator of the same meshes: shapes at
the edges of its transforms (one residue, lengths that fill or just pass a
power of two, more columns than patches, one row or layer), and a grid whose
transforms exceed a workgroup's LDS, which keeps the convolution blocks.

Both are FP64; the transforms' rounding is a few eps of the row norms, so
every component agrees to 1e-12 in norm (the bound of the other operators)."""
import numpy as np
import pytest

import oetqf_amd as oq
from helpers import relerr, rs_props, visc_props

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nxi,dip,cells,rfzh", [
    (8, 2, 90.0, (8, 3, 1), None),             # m = 1, one layer
    (9, 3, 90.0, (3, 4, 2), [1.0, 2.0]),       # m = 3
    (17, 2, 60.0, (17, 1, 2), None),           # one row, P = 64 for 33 offsets
    (16, 5, 90.0, (4, 16, 1), None),           # Py = 32 filled
    (34, 2, 90.0, (2, 17, 1), [1.0]),          # m = 17, Py = 64
    (34, 1, 90.0, (34, 34, 1), None),          # P = Py = 128: beyond the LDS
])
def test_grid_operator_matches_dense(rng, nx, nxi, dip, cells, rfzh):
    mf = oq.gen_mesh("RectOkada", 40e3, 12e3, 40e3 / nx, 12e3 / nxi, dip)
    ma = oq.hex8_box(-20e3, -7e3, -9e3, 40e3, 13e3, -12e3, *cells, rfzh=rfzh)
    pf, pa = rs_props(mf, rng), visc_props(ma, rng, 2.0)
    v = pf.vpl * np.exp(rng.standard_normal(pf.a.shape))
    u = oq.ArrayPartition(v, pf.L / v, np.zeros((ma.ne, 6)), 1e6 * rng.standard_normal((ma.ne, 6)), np.zeros(pf.a.shape))
    du = []
    for kd in ("fft_grid", "fp64"):
        p = oq.assemble_from_mesh(mf, ma, 3e10, 2e10, pf, pa, u, (0.0, 1.0), ftype=oq.DipSlip(), kdtype=kd)
        d = oq.similar(u)
        for _ in range(2):  # the second on used work buffers
            p.f(d, u, None, 0.0)
        du.append(d)
        p.f.close()
    for k in range(5):
        assert relerr(du[0].x[k], du[1].x[k]) <= 1e-12, k


@pytest.mark.parametrize("nx,nxi,cells", [(16, 4, (4, 3, 2)), (17, 2, (17, 1, 2))])
def test_spectra_take_the_tables_place(rng, nx, nxi, cells):
    """The resident operator is K_ff's kernel and the spectra alone; expanded,
    it still has the entries of the pair kernels, and the right-hand side is
    the same before and after."""
    mf = oq.gen_mesh("RectOkada", 40e3, 12e3, 40e3 / nx, 12e3 / nxi, 90.0)
    ma = oq.hex8_box(-20e3, -7e3, -9e3, 40e3, 13e3, -12e3, *cells)
    pf, pa = rs_props(mf, rng), visc_props(ma, rng, 0.0)
    v = pf.vpl * np.exp(rng.standard_normal(pf.a.shape))
    u = oq.ArrayPartition(v, pf.L / v, np.zeros((ma.ne, 6)), 1e6 * rng.standard_normal((ma.ne, 6)), np.zeros(pf.a.shape))
    p = oq.assemble_from_mesh(mf, ma, 3e10, 2e10, pf, pa, u, (0.0, 1.0), ftype=oq.DipSlip(), kdtype="fft_grid")
    a, b = oq.similar(u), oq.similar(u)
    p.f(a, u, None, 0.0)
    K, nf = p.f.dense_operator(), nx * nxi
    p.f(b, u, None, 0.0)
    nbytes = p.f.info()[2]
    p.f.close()
    mx, my, mz = cells
    m, pow2 = nx // mx, lambda n: 1 << (n - 1).bit_length()
    P, Py = pow2(2 * mx - 1), pow2(max(2, 2 * my - 1))
    bins, planes = P // 2 + 1, 6 * mz
    assert nbytes == 8 * nf * nxi + 16 * bins * (2 * planes * my * nxi * m + Py * planes ** 2)
    want = dict(fm=oq.stress_greens_function(ma, mf, 3e10, 2e10, ftype=oq.DipSlip()),
                mm=oq.stress_greens_function(ma, 3e10, 2e10, checkeigvals=False))
    for k, blk in (("fm", K[:nf, nf:]), ("mm", K[nf:, nf:])):
        assert np.abs(blk - want[k]).max() <= 1e-12 * np.abs(want[k]).max(), k
    gmf = oq.stress_greens_function(mf, ma, 3e10, 2e10, ftype=oq.DipSlip())
    assert relerr(K[nf:, :nf], gmf) <= 1e-9  # Okada's closed form from shifted coordinates
    for x, y in zip(a.x, b.x):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("kind", ["rupture", "one patch"])
def test_rates_over_many_decades_component_by_component(rng, kind):
    """Slip rates over 16 decades, and a single patch at 1 m/s on a locked
    fault: every component of the stress rates against extended-precision sums
    of the same operator.  The rounding of a transform spreads over its
    outputs, so each component is held to 64 eps (lg 64 x lg 32 butterflies, two
    passes and the products) of the largest sum |K||s| within its layer and
    stress component, not of its own."""
    nx, nxi, cells = 32, 8, (16, 12, 2)
    mf = oq.gen_mesh("RectOkada", 80e3, 20e3, 80e3 / nx, 20e3 / nxi, 90.0)
    ma = oq.hex8_box(-40e3, -20e3, -10e3, 80e3, 40e3, -30e3, *cells)
    pf, pa = rs_props(mf, rng), visc_props(ma, rng, 0.0)
    pa = oq.PowerLawViscosityProperty(pa.γ, np.zeros(ma.ne), np.zeros(6))
    shp = pf.a.shape
    if kind == "rupture":
        v = 10.0 ** rng.uniform(-16, 0, shp)
    else:
        v = np.full(shp, 1e-16)
        v[nx // 3, nxi // 2] = 1.0
    sg = 1e6 * rng.standard_normal((ma.ne, 6))
    u = oq.ArrayPartition(v, pf.L / v, np.zeros((ma.ne, 6)), sg, np.zeros(shp))
    p = oq.assemble_from_mesh(mf, ma, 3e10, 3e10, pf, pa, u, (0.0, 1.0), kdtype="fft_grid")
    K, nf, d = p.f.dense_operator(), nx * nxi, oq.similar(u)
    p.f(d, u, None, 0.0)
    p.f.close()
    dev = sg.copy()
    for k in (0, 3, 5):
        dev[:, k] -= (sg[:, 0] + sg[:, 3] + sg[:, 5]) / 3.0
    s = np.concatenate([(v - pf.vpl).ravel(order="F"), (pa.γ[:, None] * dev).ravel(order="F")])
    Km = K[nf:].astype(np.longdouble)
    ref = (Km @ s.astype(np.longdouble)).reshape((ma.ne, 6), order="F")
    size = (np.abs(Km) @ np.abs(s)).reshape((ma.ne, 6), order="F")
    layer = np.arange(ma.ne) // (cells[0] * cells[1])
    for z in range(cells[2]):
        for k in range(6):
            err = np.abs(d.x[3][layer == z, k] - ref[layer == z, k]).max()
            assert err <= 64 * np.finfo(float).eps * size[layer == z, k].max(), (z, k)
