"""oq_ensemble_eval, oq_group_eval and the timings between two stretches of a
run: the run goes on from the same states, stages and step history, so its
later states have the same bits as without them."""
import numpy as np
import pytest

import oetqf_amd as oq
from helpers import small_fault, small_mantle
from oetqf_amd.workloads import YEAR, ensemble_members

pytestmark = pytest.mark.gpu


def _model(M):
    mf, ma = small_fault(90.0, x=40e3, xi=10e3, d=2e3), small_mantle()
    shp = (mf.nx, mf.nxi)
    pf = oq.RateStateQuasiDynamicProperty(np.full(shp, 0.015), np.full(shp, 0.019), np.full(shp, 0.012),
                                          np.full(shp, 5e7), 4.9e6, 1e-9)
    pa = oq.PowerLawViscosityProperty(np.full(ma.ne, 5e-20), np.zeros(ma.ne), np.zeros(6))
    members, U = ensemble_members(dict(pf=pf, ma=ma), M, seed=5)
    return mf, ma, pa, members, U


@pytest.mark.parametrize("alg", ["tsit5", "vcabm5"])
@pytest.mark.parametrize("kind", ["ensemble", "group"])
def test_eval_and_time_leave_a_run_alone(kind, alg):
    mf, ma, pa, members, U = _model(5)
    out = []
    for look in (False, True):
        if kind == "ensemble":
            b = oq.Ensemble(mf, ma, 3e10, 3e10, members, pa, kdtype="fp32")
        else:
            b = oq.Group([(mf, ma, pa)], 3e10, 3e10, [members])
        U0 = U if kind == "ensemble" else b.pack([U])
        b.start(U0, (0.0, 100 * YEAR), dt0=1.0, alg=oq.Tsit5() if alg == "tsit5" else oq.VCABM5())
        for _ in range(3):
            b.run(7)
            if look:
                b.eval(1.5 * U0)
                b.time(2)
        out.append(b.state())
        b.close()
    for x, y in zip(out[0][:4], out[1][:4]):
        assert np.array_equal(x, y)
