"""A recorder that finds no memory: oq_stepper_record returns the error and
leaves the stepper without one, and the run goes on as an unrecorded run does,
bit for bit, not into the buffers of the recorder before."""
import numpy as np
import pytest

import oetqf_amd as oq
from helpers import rs_props, small_fault
from oetqf_amd import OetqfError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alg", [oq.Tsit5(), oq.VCABM5()], ids=["tsit5", "vcabm5"])
@pytest.mark.parametrize("persistent", [False, True])
def test_run_goes_on_without_a_recorder(rng, alg, persistent):
    mf = small_fault(90.0)
    pf = rs_props(mf, rng)
    v = pf.vpl * np.exp(0.1 * rng.standard_normal(pf.a.shape))
    u = oq.ArrayPartition(v, pf.L / v, np.zeros_like(v))
    prob = oq.assemble_from_mesh(mf, None, 3e10, 3e10, pf, None, u, (0.0, 1e9))
    end = []
    for recorded in (False, True):
        it = oq.Integrator(prob, reltol=1e-6, abstol=1e-8, alg=alg)
        it.set_persistent(persistent)
        if recorded:
            it.record(stride=1, snap_capacity=64, step_capacity=64)
        it.step(20)
        if recorded:
            with pytest.raises(OetqfError, match="hipMalloc"):
                it.record(stride=1, snap_capacity=10 ** 13, step_capacity=64)
            with pytest.raises(ValueError):
                it.drain()
        it.step(20)
        t, dt, x, na, nr = it.state()
        end.append((t, dt, na, nr, x.pack()))
        it.close()
    prob.f.close()
    for a, b in zip(*end):
        assert np.array_equal(a, b)
