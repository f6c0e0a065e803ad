"""The ensemble GEMMs' shapes: member tiles of 32, 64, 128 and 256 with the
chunks of a row sum shared out over workgroups, one chunk each (the small
models with FP32 and BF16) or several (16512 rows, tiles of up to 64), and not shared out (16512
rows, tiles of 128 and 256; 33280 rows, all tiles).  Every shape adds the same
products in the same order, so a member's derivative has the same bits whatever
the ensemble around it; and it equals the member's own FP64 right-hand side to
the FP32 operator's 2e-6 (2e-2 with the BF16 operator)."""
import numpy as np
import pytest

import oetqf_amd as oq
from helpers import relerr, small_fault, small_mantle
from oetqf_amd.workloads import ensemble_members

pytestmark = pytest.mark.gpu


def _members(mf, ma, M, rng):
    shp = (mf.nx, mf.nxi)
    pf = oq.RateStateQuasiDynamicProperty(np.full(shp, 0.015), np.full(shp, 0.019), np.full(shp, 0.012),
                                          np.full(shp, 5e7), 4.9e6, 1e-9)
    members, U = ensemble_members(dict(pf=pf, ma=ma), M, seed=5)
    if ma is not None:  # stresses off zero, so that the strain rates act
        nf = mf.nx * mf.nxi
        U[:, 2 * nf + 6 * ma.ne:2 * nf + 12 * ma.ne] = 1e6 * rng.standard_normal((M, 6 * ma.ne))
    return members, U


@pytest.mark.parametrize("kdtype", ["fp32", "fp16x2", "bf16"])
@pytest.mark.parametrize("coupled", [True, False])
def test_every_member_tile_gives_the_same_bits(rng, kdtype, coupled):
    mf, ma = small_fault(90.0, x=40e3, xi=15e3, d=1.25e3), small_mantle() if coupled else None
    pa = oq.PowerLawViscosityProperty(np.full(ma.ne, 5e-20), np.zeros(ma.ne), np.zeros(6)) if coupled else None
    members, U = _members(mf, ma, 257, rng)
    ref = None
    for M in (257, 256, 129, 128, 65, 64, 33, 32, 31, 1):
        e = oq.Ensemble(mf, ma, 3e10, 3e10, members[:M], pa, kdtype=kdtype)
        dU = e.eval(U[:M])
        e.close()
        if ref is None:
            ref = dU
        assert np.array_equal(dU, ref[:M]), M
    shp = (mf.nx, mf.nxi)
    u = oq.ArrayPartition(*([np.zeros(shp)] * 2 + ([np.zeros((ma.ne, 6))] * 2 if coupled else []) + [np.zeros(shp)]))
    for m in (0, 256):
        p = oq.assemble_from_mesh(mf, ma, 3e10, 3e10, members[m], pa, u, (0.0, 1.0))
        um, dm = oq.similar(u).unpack(U[m]), oq.similar(u)
        p.f(dm, um, None, 0.0)
        p.f.close()
        assert relerr(ref[m], dm.pack()) <= (2e-2 if kdtype == "bf16" else 2e-6), m


@pytest.mark.parametrize("kdtype", ["fp32", "fp16x2", "bf16"])
@pytest.mark.parametrize("nx,nxi", [(344, 48), (520, 64)])
def test_large_models_share_out_several_chunks_or_none(rng, kdtype, nx, nxi):
    mf = oq.gen_mesh("RectOkada", nx * 200.0, nxi * 250.0, 200.0, 250.0, 90.0)
    assert mf.nx * mf.nxi in (16512, 33280)
    members, U = _members(mf, None, 130, rng)
    U[:, :nx * nxi] *= np.exp(0.3 * rng.standard_normal((130, nx * nxi)))
    ref = None
    for M in (130, 65, 33, 2):
        e = oq.Ensemble(mf, None, 3e10, 3e10, members[:M], None, kdtype=kdtype)
        dU = e.eval(U[:M])
        e.close()
        if ref is None:
            ref = dU
        assert np.array_equal(dU, ref[:M]), M
    shp = (mf.nx, mf.nxi)
    u = oq.ArrayPartition(*[np.zeros(shp) for _ in range(3)])
    for m in (0, 129):  # by DFT: the FP64 operator without its dense rows
        p = oq.assemble_from_mesh(mf, None, 3e10, 3e10, members[m], None, u, (0.0, 1.0), kdtype="fft")
        um, dm = oq.similar(u).unpack(U[m]), oq.similar(u)
        p.f(dm, um, None, 0.0)
        p.f.close()
        assert relerr(ref[m], dm.pack()) <= (2e-2 if kdtype == "bf16" else 2e-6), m
