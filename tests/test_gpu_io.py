"""Uploads and downloads of FP32 fields, through the C ABI with pageable and
pinned arrays: the values that come back are the FP64 ones rounded to FP32
once, bit for bit, whichever side converts them.  Sizes: below and above the
2^21 values from which pageable arrays are converted on the device, one point
past its buffer of 2^22 values, and ragged ones."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 16), (33, 31, 21), (128, 128, 128), (127, 129, 131), (161, 162, 161)]


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_fp32_roundtrip(shape, pinned):
    import torch

    import cosmograph_amd as cg
    print(f"case io shape={shape} pinned={pinned}", flush=True)
    g = cg.BSSN(cg.GpuParams(n=shape, order=4, precision="fp32_split"))
    rng = np.random.default_rng(7)
    a = rng.standard_normal(shape) * 10.0 ** rng.integers(-44, 30, size=shape)
    a.reshape(-1)[:4] = [np.inf, -np.inf, np.nan, -0.0]
    n = a.size
    up = torch.empty(shape, dtype=torch.float64, pin_memory=pinned)
    down = torch.empty(shape, dtype=torch.float64, pin_memory=pinned)
    up.copy_(torch.from_numpy(a))
    down.fill_(5.0)
    ptr = lambda t: ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))  # noqa: E731
    assert g.L.cg_field_upload(g.h, b"A12_p", ptr(up), n) == 0
    assert g.L.cg_field_download(g.h, b"A12_p", ptr(down), n) == 0
    with np.errstate(over="ignore"):
        want = a.astype(np.float32).astype(np.float64)
    np.testing.assert_array_equal(down.numpy(), want)
    assert np.signbit(down.numpy().reshape(-1)[3])
    assert np.count_nonzero(g.download("A11_p")) == 0
    assert np.count_nonzero(g.download("A13_p")) == 0
