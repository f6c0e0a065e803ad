"""The dense matvec's rows per wavefront (one, two, four or eight by rows and
type): at the ends of each choice, with ragged last workgroups, the fault-only
right-hand side is the DFT operator's, which has no dense rows: to 1e-12 with
the FP64 operator, 1e-5 with FP32 and 2e-2 with BF16, as elsewhere."""
import numpy as np
import pytest

import oetqf_amd as oq
from helpers import relerr, rs_props, small_fault

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nxi", [(1, 1), (5, 3), (40, 32), (61, 21), (64, 40), (197, 13), (87, 89), (128, 64),
                                    (257, 32), (211, 58), (197, 32), (199, 32), (205, 40), (260, 32), (330, 32),
                                    (395, 32)])
def test_rows_per_wavefront(rng, nx, nxi):
    mf = small_fault(90.0, x=nx * 1e3, xi=nxi * 1e3, d=1e3)
    assert (mf.nx, mf.nxi) == (nx, nxi)
    pf = rs_props(mf, rng)
    v = pf.vpl * np.exp(0.3 * rng.standard_normal((nx, nxi)))
    u = oq.ArrayPartition(v, pf.L / v, np.zeros_like(v))
    out = {}
    for kd in ("fft", "fp64", "fp32", "bf16"):
        p = oq.assemble_from_mesh(mf, None, 3e10, 3e10, pf, None, u, (0.0, 1.0), kdtype=kd)
        d = oq.similar(u)
        p.f(d, u, None, 0.0)
        p.f.close()
        out[kd] = d
    for kd, tol in (("fp64", 1e-12), ("fp32", 1e-5), ("bf16", 2e-2)):
        assert relerr(out[kd].x[0], out["fft"].x[0]) <= tol, kd
        for a, b in zip(out[kd].x[1:], out["fft"].x[1:]):
            assert np.array_equal(a, b), kd
