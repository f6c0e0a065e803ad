"""Models of different sizes alive at once: what a small one sets up for the
kernels that both use (the limit on their LDS belongs to the function) leaves
the large one's next evaluation as it was, bit for bit."""
import numpy as np
import pytest

import oetqf_amd as oq
from helpers import rs_props, visc_props

pytestmark = pytest.mark.gpu

#        kdtype, (nx, nxi, mantle cells) of the large model: over 64 KB of LDS per workgroup, and of the small one
CASES = {
    "grid in the frequency domain": ("fft_grid", (32, 2, (32, 34, 1)), (8, 2, (4, 2, 1))),
    "grid convolution blocks": ("fft_grid", (34, 1, (34, 50, 1)), (9, 2, (2, 2, 1))),
    "DFT": ("fft", (1500, 1, None), (16, 2, None)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_a_small_model_leaves_a_large_one_alone(rng, name):
    kd, large, small = CASES[name]

    def model(nx, nxi, cells):
        mf = oq.gen_mesh("RectOkada", 40e3, 12e3, 40e3 / nx, 12e3 / nxi, 90.0)
        ma = oq.hex8_box(-20e3, -7e3, -9e3, 40e3, 13e3, -12e3, *cells) if cells else None
        pf = rs_props(mf, rng)
        v = pf.vpl * np.exp(rng.standard_normal(pf.a.shape))
        m = [np.zeros((ma.ne, 6)), 1e6 * rng.standard_normal((ma.ne, 6))] if cells else []
        u = oq.ArrayPartition(v, pf.L / v, *m, np.zeros(pf.a.shape))
        pa = visc_props(ma, rng, 0.0) if cells else None
        return oq.assemble_from_mesh(mf, ma, 3e10, 2e10, pf, pa, u, (0.0, 1.0), kdtype=kd), u

    p, u = model(*large)
    a, b = oq.similar(u), oq.similar(u)
    p.f(a, u, None, 0.0)
    q, w = model(*small)
    d = oq.similar(w)
    q.f(d, w, None, 0.0)
    p.f(b, u, None, 0.0)
    q.f.close()
    p.f.close()
    for x, y in zip(a.x, b.x):
        assert np.all(np.isfinite(x)) and np.array_equal(x, y)
