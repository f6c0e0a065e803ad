"""Operator blocks that closed models leave for the next one: a model built in
blocks full of NaN is, bit for bit, the one built in fresh memory (every block
is written in full or cleared, the padding of its rows included), and
oq_release_memory and the creation of a batch give the blocks back."""
import ctypes

import numpy as np
import pytest

import oetqf_amd as oq
from helpers import rs_props, visc_props
from oetqf_amd import _lib

pytestmark = pytest.mark.gpu
MB = 1 << 20


def _free():
    """Free device memory, from the HIP runtime that the library is linked with."""
    _lib.load()
    rt = ctypes.CDLL("libamdhip64.so.7")
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert rt.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


def _ld(n):
    return (n + 511) // 512 * 512


def _fault(nx, nxi, rng):
    mf = oq.gen_mesh("RectOkada", nx * 1e3, nxi * 5e2, 1e3, 5e2, 90.0)
    assert (mf.nx, mf.nxi) == (nx, nxi)
    pf = rs_props(mf, rng)
    v = pf.vpl * np.exp(0.3 * rng.standard_normal((nx, nxi)))
    return mf, pf, v


def _leave_nan_blocks(sizes, rng):
    """Closed models whose FP64 operators, all NaN, fit allocations of these sizes; their bytes."""
    models, total = [], 0
    for s in sizes:
        n = 512
        while n * _ld(n) * 8 < 1.03 * s:  # another N: the padding lies elsewhere
            n += 2
        assert n * _ld(n) * 8 <= 1.12 * s, "no block for %d bytes" % s
        _, pf, v = _fault(n // 2, 2, rng)
        p = oq.assemble(np.full((n // 2, 2, 2), np.nan), pf, oq.ArrayPartition(v, pf.L / v, np.zeros_like(v)), (0.0, 1.0))
        d = oq.ArrayPartition(*[np.zeros_like(v) for _ in range(3)])
        p.f(d, oq.ArrayPartition(v, pf.L / v, np.zeros_like(v)), None, 0.0)
        assert np.all(np.isnan(d.x[0]))
        models.append(p)
        total += n * _ld(n) * 8
    for p in models:
        p.f.close()
    return total


N, LD = 4300, 4608
CASES = {  # kdtype, fault, mantle cells, the blocks its assembly takes
    "fp64": ((86, 50), None, [N * LD * 8]),
    "fp32": ((86, 50), None, [N * LD * 8, N * LD * 4]),
    "bf16": ((86, 50), None, [N * LD * 8, N * LD * 2]),
    "coupled fp64": ((38, 50), (10, 10, 4), [N * LD * 8]),
    "coupled fft": ((38, 50), (10, 10, 4), [2400 * LD * 8, 1900 * 2560 * 8]),
    # the tables along strike (three blocks) and the spectra of K_fm and K_mf
    "coupled fft_grid": ((128, 30), (16, 16, 8), [768 * 30 * 248 * 8] * 3 + [17 * 768 * 240 * 16] * 2),
}


@pytest.mark.parametrize("name", list(CASES))
def test_recycled_blocks_hold_nothing_of_the_last_model(rng, name):
    (nx, nxi), cells, sizes = CASES[name]
    mf, pf, v = _fault(nx, nxi, rng)
    ma = pa = None
    m = []
    if cells:
        ma = oq.hex8_box(-nx * 5e2, -8e3, -30e3, nx * 1e3, 16e3, -12e3, *cells)
        pa = visc_props(ma, rng, 0.0)
        m = [np.zeros((ma.ne, 6)), 1e6 * rng.standard_normal((ma.ne, 6))]
    u = oq.ArrayPartition(v, pf.L / v, *m, np.zeros_like(v))
    out = []
    for blocks in ([], sizes):
        oq.release_memory()
        left = _leave_nan_blocks(blocks, rng)
        p = oq.assemble_from_mesh(mf, ma, 3e10, 2e10, pf, pa, u, (0.0, 1.0), kdtype=name.split()[-1])
        before = _free()
        oq.release_memory()  # what the model has not taken
        unused = _free() - before
        d = oq.similar(u)
        p.f(d, u, None, 0.0)
        p.f.close()
        out.append(d)
    assert unused < left - 0.9 * sizes[-1], "the second model was not built in the kept blocks"
    for a, b in zip(out[0].x, out[1].x):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
    oq.release_memory()


def test_release_memory_gives_the_blocks_back(rng):
    mf, pf, v = _fault(86, 50, rng)
    u = oq.ArrayPartition(v, pf.L / v, np.zeros_like(v))
    oq.assemble_from_mesh(mf, None, 3e10, 2e10, pf, None, u, (0.0, 1.0)).f.close()
    oq.release_memory()
    start = _free()
    oq.assemble_from_mesh(mf, None, 3e10, 2e10, pf, None, u, (0.0, 1.0)).f.close()
    kept = start - _free()
    assert abs(kept - N * LD * 8) <= 16 * MB  # the runtime's own pages on either side
    oq.release_memory()
    assert abs(start - _free()) <= 16 * MB


@pytest.mark.parametrize("kind", ["fp16x2", "fp32", "group"])
def test_a_batch_leaves_no_blocks_beside_it(rng, kind):
    mf, pf, v = _fault(86, 50, rng)
    oq.release_memory()
    if kind == "group":
        b = oq.Group([(mf, None, None)], 3e10, 2e10, [[pf] * 3])
    else:
        b = oq.Ensemble(mf, None, 3e10, 2e10, [pf] * 3, None, kdtype=kind)
    alive = _free()
    oq.release_memory()
    assert _free() - alive <= 16 * MB
    b.close()
    oq.release_memory()
