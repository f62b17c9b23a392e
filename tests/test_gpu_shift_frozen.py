"""Fused steps of every shift gauge that has them with a lapse identically 1
(Static lapse, DIFFalpha zero: nothing of the lapse is staged, also not for the
DampedWave shift, whose beta equation has its gradient), against the method
sequence.  Bars: FP64 1e-12 relative L2, as tests/test_gpu_shift_fused.py;
split precision 2e-5, twice the 1e-5 that each form is from the oracle."""
import numpy as np
import pytest

from common import FIELDS, rel_l2
from test_gpu_shift import shift_state, x_fields

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import cosmograph_amd as cg
    cg.load_library()
    return cg


@pytest.mark.parametrize("prec", ["fp64", "fp32_split"])
@pytest.mark.parametrize("order,shape", [(2, (17, 13, 20)), (4, (18, 14, 20)), (6, (9, 11, 36))])
@pytest.mark.parametrize("shift", ["DampedWave", "GammaDriver", "Static", "AwAShiftedWave"])
def test_frozen_lapse(gpu, shift, order, shape, prec):
    print(f"case frozen lapse {shift} order {order} {shape} {prec}", flush=True)
    st = shift_state(shape, 5)
    st["DIFFalpha"][:] = 0.0
    names = FIELDS + x_fields(shift)
    runs = []
    for fused in (True, False):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=order, precision=prec, lapse="Static", shift=shift, matter="static",
                                   gauge_wave_dir=2, gd_eta=0.4, dw_mu_s=0.3, dw_mu_l=0.2, dw_p=0.5))
        g.set_dma(fused)
        for f in names:
            g.upload(f + "_p", st[f])
        g.upload("DIFFD_a", st["DIFFD"])
        g.frw_set(0.0, -3.0)
        g.frw_add_fluid(3.0 / (8.0 * np.pi), 0.0)
        g.step(3)
        runs.append({f: g.download(f + "_p") for f in names})
    tol = 1e-12 if prec == "fp64" else 2e-5
    for f in names:
        assert rel_l2(runs[0][f], runs[1][f]) <= tol, f
    assert np.count_nonzero(runs[0]["DIFFalpha"]) == 0
