"""LDS-DMA staging in FP64 on grids whose nz is a multiple of 2 but not of 4.

Rows are whole 16-byte groups there too (two FP64 values), so the DMA kernels
of the stages, of the constraints and of the shift build's gauge terms run;
set_dma(False) gives the register-staged kernels, or the method sequence of the
shift build, on the same grid.  nz sits 2 past a tile, 2 before one and at the
smallest value that the 16-point tile takes (20 for a halo rounded up to 4).
Bars, derived before the first run: the same arithmetic in both kernels, apart
from the compiler's contractions of multiply-adds, through 8 stage evaluations
of about 10 roundings of 1.1e-16: 1e-14 relative L2.  The shift's method
sequence orders its sums differently and the dust is compared with the oracle:
1e-12, the bar of their own tests.  A wrong halo element
is many orders of magnitude off."""
import numpy as np
import pytest

from common import FIELDS, rel_l2, smooth_random_state
from test_gpu_dust import check, dust_pair
from test_gpu_shift import X_ALL, shift_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import cosmograph_amd as cg
    cg.load_library()
    return cg


def _start(g, st, fields):
    for f in fields:
        g.upload(f + "_p", st[f])
    g.upload("DIFFD_a", st["DIFFD"])
    g.frw_set(0.0, -3.0)
    g.frw_add_fluid(3.0 / (8.0 * np.pi), 0.0)


STAGE = [(2, (17, 13, 22), "Static", 0.0), (2, (16, 12, 34), "Harmonic", 0.2), (4, (17, 13, 22), "Static", 0.0),
         (4, (8, 12, 30), "OnePlusLog", 0.0), (6, (18, 14, 34), "Static", 0.0), (6, (16, 16, 22), "Harmonic", 0.0),
         (8, (16, 16, 26), "Static", 0.0), (8, (18, 17, 22), "Harmonic", 0.1)]


@pytest.mark.parametrize("order,shape,lapse,ko", STAGE)
def test_stages(gpu, order, shape, lapse, ko):
    print(f"case even dma order {order} {shape} {lapse} ko {ko}", flush=True)
    st = smooth_random_state(shape, seed=order, with_alpha=lapse != "Static")
    out, lds = [], []
    for dma in (True, False):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=order, lapse=lapse, ko_coeff=ko))
        g.set_dma(dma)
        _start(g, st, FIELDS)
        g.step(2)
        out.append({f: g.download(f + "_p") for f in FIELDS})
        lds.append(g.kernel_info()["lds_bytes"])
    assert lds[0] != lds[1]  # the DMA kernel ran
    for f in FIELDS:
        assert rel_l2(out[0][f], out[1][f]) <= 1e-14, f


@pytest.mark.parametrize("order,shape,lapse,norm", [(4, (17, 13, 22), "Static", 1), (4, (16, 12, 50), "Harmonic", 1),
                                                    (6, (18, 14, 34), "Static", 1), (6, (9, 11, 30), "OnePlusLog", 1),
                                                    (6, (16, 16, 22), "Static", 0)])
def test_split_stages(gpu, order, shape, lapse, norm):
    """FP32 split: the FP64 metric moves in pairs, the FP32 fields in single
    words.  Bar: that of the DMA test in split precision (1e-7)."""
    print(f"case even dma split order {order} {shape} {lapse} norm {norm}", flush=True)
    st = smooth_random_state(shape, seed=order + 1, with_alpha=lapse != "Static")
    out, info = [], []
    for dma in (True, False):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=order, lapse=lapse, precision="fp32_split", normalize_metric=norm))
        g.set_dma(dma)
        _start(g, st, FIELDS)
        g.step(3)
        out.append({f: g.download(f + "_p") for f in FIELDS})
        info.append(g.kernel_info())
    assert info[0] != info[1]  # the DMA kernel ran
    for f in FIELDS:
        assert rel_l2(out[0][f], out[1][f]) <= 1e-7, f


@pytest.mark.parametrize("order,shape", [(4, (17, 13, 22)), (6, (18, 14, 34))])
def test_constraints(gpu, order, shape):
    print(f"case even dma constraints order {order} {shape}", flush=True)
    st = smooth_random_state(shape, seed=9)
    res = []
    for dma in (True, False):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=order))
        g.set_dma(dma)
        _start(g, st, FIELDS)
        g.stepInit()
        res.append(g.setConstraintCalcs())
    for k in ("H", "M"):
        a, b = np.array(res[0][k]), np.array(res[1][k])
        assert np.all(np.abs(a - b) <= 1e-12 * np.abs(b) + 1e-14), (k, a, b)


@pytest.mark.parametrize("order,shape", [(4, (18, 14, 22)), (6, (9, 11, 34)), (2, (16, 16, 30))])
def test_fused_shift_steps(gpu, order, shape):
    print(f"case even dma shift order {order} {shape}", flush=True)
    st = shift_state(shape, 5)
    out = []
    for dma in (True, False):
        g = gpu.BSSN(gpu.GpuParams(n=shape, order=order, lapse="OnePlusLog", shift="GammaDriver", gd_eta=0.4))
        g.set_dma(dma)
        _start(g, st, FIELDS + X_ALL)
        g.step(3)
        out.append({f: g.download(f + "_p") for f in FIELDS + X_ALL})
    for f in out[0]:
        assert rel_l2(out[0][f], out[1][f]) <= 1e-12, f


@pytest.mark.parametrize("order,shape", [(4, (18, 16, 22)), (4, (17, 13, 34)), (6, (18, 14, 30))])
def test_dust(oracle_mod, gpu, order, shape):
    print(f"case even dma dust order {order} {shape}", flush=True)
    o, g = dust_pair(oracle_mod, gpu, shape, order)
    o.run_steps(2)
    g.step(2)
    info = g.kernel_info()
    check(g, o, tol=1e-12)
    g.set_dma(False)
    assert info != g.kernel_info()  # the DMA kernel ran (4x8x8 at order 4: the same LDS size, other registers)
