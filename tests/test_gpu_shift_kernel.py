"""Which kernels run: fused steps of the shift build report a NaN that the last
step of a call produced, which the method sequence leaves to the next call, and
kernel_info names their 4x4x16 stage kernel; the two forms of the constraint
kernel split the grid into other tiles, so their sums differ in the last bits.
These hold for the contexts of the tests that compare the forms with each
other, which would pass if both sides ran the same one."""
import numpy as np
import pytest

from common import FIELDS, rel_l2, smooth_random_state
from test_gpu_shift_fused import CASES as FUSED
from test_gpu_dma_even import _start
from test_gpu_shift import X_ALL, shift_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import cosmograph_amd as cg
    cg.load_library()
    return cg


def steps_fused(gpu, g):
    """Whether the next step is a fused one (the state is lost)."""
    k = g.download("DIFFK_p")
    k[5, 6, 7] = np.nan
    g.upload("DIFFK_p", k)
    try:
        g.step(1)
    except gpu.CosmoGpuError as e:
        assert e.code == gpu.ERR_NAN
        return True
    return False


def infos(gpu, shape, shift, order, lapse, prec="fp64", ko=0.0):
    """kernel_info of the shift context (DMA staging on, off) and of a context
    without a shift on the same grid, and whether the shift ones step fused."""
    def one(s, dma):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=order, lapse=lapse, shift=s, precision=prec, ko_coeff=ko))
        if lapse == "Static":
            g.upload("DIFFalpha_p", np.full(shape, 1e-3))  # as the tests that use these cases: a lapse that is not 1
        g.set_dma(dma)
        return g.kernel_info(), s != "none" and steps_fused(gpu, g)
    (on, f_on), (off, f_off) = one(shift, True), one(shift, False)
    return on, off, one("none", True)[0], one("none", False)[0], f_on, f_off


# the tests of the fused steps
EVEN = [((18, 14, 22), "GammaDriver", 4, "OnePlusLog", "fp64", 0.0), ((9, 11, 34), "GammaDriver", 6, "OnePlusLog", "fp64", 0.0),
        ((16, 16, 30), "GammaDriver", 2, "OnePlusLog", "fp64", 0.0)]
REGISTERS = [((18, 14, 20), "GammaDriver", 4, "OnePlusLog", "fp64", 0.0), ((18, 14, 20), "Static", 4, "OnePlusLog", "fp64", 0.0)]


@pytest.mark.parametrize("shape,shift,order,lapse,prec,ko", FUSED + EVEN + REGISTERS)
def test_fused_kernel_runs(gpu, shape, shift, order, lapse, prec, ko):
    on, off, plain_on, plain_off, f_on, f_off = infos(gpu, shape, shift, order, lapse, prec, ko)
    assert f_on and not f_off
    assert on["tile"] == (4, 4, 16)
    assert off == plain_off


def test_fused_kernel_of_a_frozen_lapse(gpu):
    for dma in (True, False):
        g = gpu.BSSN(gpu.GpuParams(n=(18, 14, 20), order=4, lapse="Static", shift="GammaDriver", normalize_metric=0))
        g.set_dma(dma)
        assert not dma or g.kernel_info()["tile"] == (4, 4, 16)
        assert steps_fused(gpu, g) == dma


# other fields' complete right-hand sides; a halo of 4; rows that are no whole 16-byte groups; fewer points than a tile needs
@pytest.mark.parametrize("shape,shift,order,lapse,prec", [((18, 14, 20), "AijDriverShift", 4, "OnePlusLog", "fp64"),
                                                          ((18, 14, 20), "GammaDriver", 4, "TestKDriverLapse", "fp64"),
                                                          ((18, 18, 24), "GammaDriver", 8, "OnePlusLog", "fp64"),
                                                          ((18, 14, 21), "GammaDriver", 4, "OnePlusLog", "fp64"),
                                                          ((18, 14, 22), "GammaDriver", 4, "OnePlusLog", "fp32_split"),
                                                          ((18, 14, 18), "GammaDriver", 4, "OnePlusLog", "fp64")])
def test_no_fused_kernel(gpu, shape, shift, order, lapse, prec):
    on, off, plain_on, plain_off, f_on, f_off = infos(gpu, shape, shift, order, lapse, prec)
    assert not f_on and not f_off
    assert on == plain_on and off == plain_off


@pytest.mark.parametrize("order,shape,dma_form", [(4, (17, 13, 22), True), (6, (18, 14, 34), True), (4, (17, 13, 21), False)])
def test_constraint_forms(gpu, order, shape, dma_form):
    st = smooth_random_state(shape, seed=9)
    res = []
    for dma in (True, False):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=order))
        g.set_dma(dma)
        _start(g, st, FIELDS)
        g.stepInit()
        res.append(g.setConstraintCalcs())
    equal = all(np.array_equal(res[0][k], res[1][k]) for k in ("H", "M", "G"))
    assert equal == (not dma_form)


def test_requested_tile(gpu):
    """A tile asked for at creation is the one that runs (the method sequence
    where the fused steps have no such tile), or an error where nothing has it."""
    shape, st = (18, 14, 20), shift_state((18, 14, 20), 5)

    def ctx(tile, shift="GammaDriver"):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=4, lapse="OnePlusLog", shift=shift, gd_eta=0.4, tile=tile))
        _start(g, st, FIELDS + (X_ALL if shift != "none" else []))
        return g

    fused = ctx((4, 4, 16)).kernel_info()
    assert fused == ctx((0, 0, 0)).kernel_info() and fused["tile"] == (4, 4, 16)
    assert steps_fused(gpu, ctx((4, 4, 16))) and not steps_fused(gpu, ctx((4, 8, 8)))
    g = ctx((4, 8, 8))
    assert g.kernel_info() == ctx((4, 8, 8), "none").kernel_info()
    g.step(2)
    h = ctx((0, 0, 0))
    h.set_dma(False)  # the method sequence
    h.step(2)
    for f in FIELDS + X_ALL:
        assert rel_l2(g.download(f + "_p"), h.download(f + "_p")) <= 1e-12, f
    for shift in ("none", "GammaDriver"):
        with pytest.raises(gpu.CosmoGpuError) as e:
            ctx((4, 4, 4), shift).step(1)
        assert e.value.code == -1  # CG_ERR_ARG
    # the autotuner's pick is no request
    a = ctx((0, 0, 0))
    a.autotune(1)
    assert a.kernel_info() == fused and steps_fused(gpu, a)
