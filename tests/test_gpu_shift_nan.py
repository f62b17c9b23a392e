"""The NaN guard of the shift build (sims/sim.cc:179-183, checked before every
step): a step does not change a state whose DIFFphi holds a NaN, fused
(LDS-DMA staging on) as in the method sequence.  The refused call leaves _p,
the shift registers and the FRW values of the last good step, and _a and _f as
stepInit leaves them.  Bar for the values of the two forms: 1e-11 relative L2
(they agree to 1e-12 per step); NaN at the same points."""
import numpy as np
import pytest

from common import FIELDS, rel_l2
from test_gpu_shift import X_ALL, shift_state
from test_gpu_shift_registers import context

pytestmark = pytest.mark.gpu

SHAPE = (18, 14, 20)


@pytest.fixture(scope="module")
def gpu():
    import cosmograph_amd as cg
    cg.load_library()
    return cg


def refused(gpu, g, n):
    with pytest.raises(gpu.CosmoGpuError) as e:
        g.step(n)
    assert e.value.code == gpu.ERR_NAN


def state(g):
    return {f + r: g.download(f + r) for f in FIELDS + X_ALL for r in ("_p", "_a", "_f")}, g.frw_get()


def same(a, b):
    assert a[1] == b[1]
    for k in b[0]:
        nan = np.isnan(b[0][k])
        assert np.array_equal(np.isnan(a[0][k]), nan), k
        assert rel_l2(np.where(nan, 0, a[0][k]), np.where(nan, 0, b[0][k])) <= 1e-11, k


@pytest.mark.parametrize("steps_before", [0, 2])
def test_state_with_a_nan_is_refused(gpu, steps_before):
    st = shift_state(SHAPE, 6)
    out = []
    for fused in (True, False):
        g = context(gpu, fused, st)
        g.step(steps_before)
        phi = g.download("DIFFphi_p")
        phi[3, 4, 5] = np.nan
        g.upload("DIFFphi_p", phi)
        want = {f: g.download(f + "_p") for f in FIELDS + X_ALL}
        frw = g.frw_get()
        for n in (3, 1):
            refused(gpu, g, n)
            for f in want:
                assert np.array_equal(g.download(f + "_p"), want[f], equal_nan=True), f
            assert g.frw_get() == frw
        # the context goes on once the state is good again
        out.append(state(g))
        phi[3, 4, 5] = 0.0
        g.upload("DIFFphi_p", phi)
        g.step(2)
        out.append((state(g)[0], g.frw_get()))
        assert np.all(np.isfinite(out[-1][0]["DIFFphi_p"]))
    same(out[0], out[2])
    a, b = ({k: v for k, v in o[0].items() if k.endswith("_p")} for o in (out[1], out[3]))
    same((a, out[1][1]), (b, out[3][1]))


def test_stops_at_the_step_that_produced_one(gpu):
    """A NaN in DIFFK reaches DIFFphi in the first step: the second is refused."""
    st = shift_state(SHAPE, 7)
    st["DIFFK"][8, 6, 9] = np.nan
    out = []
    for fused in (True, False):
        g = context(gpu, fused, st)
        refused(gpu, g, 4)
        out.append(state(g))
        assert g.numNaNs("DIFFphi_p") > 0
        refused(gpu, g, 1)
        again = state(g)
        assert again[1] == out[-1][1]
        for k in again[0]:
            assert np.array_equal(again[0][k], out[-1][0][k], equal_nan=True), k
    same(out[0], out[1])
