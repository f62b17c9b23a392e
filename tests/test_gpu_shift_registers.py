"""The registers of the shift build after fused steps, against the method
sequence that these steps stand for (run where LDS-DMA staging is off): what
the calls between steps read, write and leave behind.  Bars: the two forms
agree to 1e-12 relative L2 per step (tests/test_gpu_shift_fused.py); 1e-11 for
the registers a few calls later, 1e-10 for right-hand sides, which differentiate
them."""
import numpy as np
import pytest

from common import FIELDS, rel_l2, smooth_random_state
from test_gpu_shift import X_ALL, shift_state

pytestmark = pytest.mark.gpu

SHAPE, ORDER = (18, 14, 20), 4


@pytest.fixture(scope="module")
def gpu():
    import cosmograph_amd as cg
    cg.load_library()
    return cg


def context(gpu, fused, st, **kw):
    par = dict(n=SHAPE, order=ORDER, lapse="OnePlusLog", shift="GammaDriver", gd_eta=0.4)
    par.update(kw)
    g = gpu.BSSN(gpu.GpuParams(**par))
    g.set_dma(fused)
    for f in FIELDS + (X_ALL if par["shift"] == "GammaDriver" else X_ALL[:4]):
        g.upload(f + "_p", st[f])
    g.upload("DIFFD_a", st["DIFFD"])
    g.frw_set(0.0, -3.0)
    g.frw_add_fluid(3.0 / (8.0 * np.pi), 0.0)
    return g


def registers(g, regs="pafc"):
    return {f + "_" + r: g.download(f + "_" + r) for f in ("DIFFgamma12", "DIFFphi", "A12", "DIFFK", "beta2", "auxB1")
            for r in regs}


def same(got, want, tol=1e-11):
    for k in want:
        assert rel_l2(got[k], want[k]) <= tol, (k, rel_l2(got[k], want[k]))


def test_no_steps_change_nothing(gpu):
    """cg_rk4_steps of no steps after fused steps whose _a was written: the
    method calls that follow work on the registers as they were."""
    st = shift_state(SHAPE, 5)
    out = []
    for fused in (True, False):
        g = context(gpu, fused, st)
        g.step(1)
        g.upload("DIFFK_a", st["DIFFK"])
        g.step(0)
        g.RKEvolve()
        g.K1Finalize()
        out.append(registers(g))
    same(out[0], out[1], 1e-10)


@pytest.mark.parametrize("shift", ["none", "GammaDriver"])
def test_no_steps_keep_averages(gpu, shift):
    """The averages of the last step's K4Finalize are formed on demand: a call of
    no steps in between does not lose them."""
    st = shift_state(SHAPE, 5) if shift != "none" else smooth_random_state(SHAPE, seed=5)
    ext = []
    for zero in (False, True):
        g = gpu.BSSN(gpu.GpuParams(n=SHAPE, order=ORDER, lapse="Harmonic", shift=shift))
        for f in FIELDS + (X_ALL if shift != "none" else []):
            g.upload(f + "_p", st[f])
        g.upload("DIFFD_a", st["DIFFD"])
        before = g.extra_field_data()
        g.step(2)
        if zero:
            g.step(0)
        ext.append(g.extra_field_data())
        assert ext[-1] != before
    assert ext[0] == ext[1]
