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


def evaluations(g):
    """What is formed from _a and _f after the state changed under them."""
    c = g.setConstraintCalcs()
    spec = g.power_spectrum("DIFFphi_a")
    regs = registers(g, "pa")
    g.RKEvolve()
    regs.update(registers(g, "c"))
    g.K1Finalize()
    regs.update({k + " K1": v for k, v in registers(g, "fc").items()})
    return c, spec, regs


def compare_evaluations(a, b):
    # H and M are about 1e-3 of the terms they are the difference of
    for k in ("H", "M"):
        assert np.all(np.abs(np.array(a[0][k]) - np.array(b[0][k])) <= 1e-8 * np.abs(b[0][k])), k
    assert np.all(np.abs(a[1] - b[1]) <= 1e-10 * np.abs(b[1]) + 1e-18 * np.abs(b[1]).max())
    same(a[2], b[2], 1e-10)


def test_upload_of_p_leaves_a_and_f(gpu):
    """An upload to _p between steps changes neither _a nor _f nor what is
    evaluated from them."""
    st, other = shift_state(SHAPE, 5), shift_state(SHAPE, 8)
    out = []
    for fused in (True, False):
        g = context(gpu, fused, st)
        g.step(2)
        for f in ("DIFFK", "DIFFphi", "beta2"):
            g.upload(f + "_p", other[f])
        ev = evaluations(g)
        g.step(1)
        out.append((ev, registers(g, "p")))
    compare_evaluations(out[0][0], out[1][0])
    same(out[0][1], out[1][1])


def test_device_initial_data_leave_a_and_f(gpu):
    """The device initial data write _p registers: _a, _f and what is evaluated
    from them stay those of the last step."""
    st = shift_state(SHAPE, 5)
    nx, ny, nz = SHAPE
    rng = np.random.default_rng(3)
    modes = np.zeros((nx, ny, nz // 2 + 1), dtype=complex)
    modes[1:3, 1:3, 1:3] = rng.standard_normal((2, 2, 2)) + 1j * rng.standard_normal((2, 2, 2))
    out = []
    for fused in (True, False):
        g = context(gpu, fused, st)
        g.step(2)
        g.ics_static_dust(modes, 1e-3)
        ev = evaluations(g)
        g.step(1)
        out.append((ev, registers(g, "p")))
    compare_evaluations(out[0][0], out[1][0])
    same(out[0][1], out[1][1])


def test_step_init_keeps_c(gpu):
    """stepInit writes _a and _f: _c holds what the last step left there."""
    st = shift_state(SHAPE, 5)
    out = []
    for fused in (True, False):
        g = context(gpu, fused, st)
        g.step(2)
        before = registers(g, "c")
        g.stepInit()
        after = registers(g, "c")
        for k in before:
            assert np.array_equal(before[k], after[k]), k
        regs = registers(g, "pafc")
        for fin in (g.K1Finalize, g.K2Finalize, g.K3Finalize, g.K4Finalize):
            g.RKEvolve()
            fin()
        g.step(1)
        out.append((regs, registers(g, "pc")))
    same(out[0][0], out[1][0])
    same(out[0][1], out[1][1])
