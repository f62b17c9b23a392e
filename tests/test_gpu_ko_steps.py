"""Whole steps with Kreiss-Oliger dissipation (orders 2 and 8, the only ones
the reference has it at) and metric normalisation against the oracle: the
normalised copy materialised before the first step and, with LDS-DMA staging,
written by stage 4 for the next ones; in both RK4 forms; on grids that the DMA
path takes and on ragged ones that it does not.  Bars: FP64 1e-12 relative L2
(absolute for a zero field), FP32 split 1e-5, as for the steps without KO."""
import numpy as np
import pytest

from common import FIELDS, rel_l2, setup_pair, smooth_random_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import cosmograph_amd as cg
    cg.load_library()
    return cg


@pytest.mark.parametrize("keep", [False, True])
@pytest.mark.parametrize("shape", [(20, 24, 32), (18, 14, 21)])
@pytest.mark.parametrize("order,ko,lapse,prec", [(2, 0.3, "Static", "fp64"), (8, 0.05, "Harmonic", "fp64"),
                                                 (8, 0.05, "OnePlusLog", "fp64"), (2, 0.3, "Harmonic", "fp32_split"),
                                                 (8, 0.05, "Static", "fp32_split")])
def test_ko_steps(oracle_mod, gpu, order, ko, lapse, prec, shape, keep):
    print(f"case ko steps order={order} lapse={lapse} {prec} {shape} keep={keep}", flush=True)
    st = smooth_random_state(shape, seed=order, amp=1e-3, with_alpha=lapse != "Static")
    o, g = setup_pair(oracle_mod, gpu, {"n": shape, "order": order, "ko": ko, "lapse": lapse, "precision": prec},
                      state=st)
    g.set_fused_accumulator(keep)
    o.run_steps(3)
    g.step(2)
    g.step(1)
    tol = 1e-12 if prec == "fp64" else 1e-5
    for f in FIELDS:
        assert rel_l2(g.download(f + "_p"), o.field(f + "_p")) <= tol, f
        if prec == "fp64" and not keep:
            assert rel_l2(g.download(f + "_c"), o.field(f + "_c")) <= tol, f
    assert np.all(np.isfinite(g.download("DIFFphi_p")))
