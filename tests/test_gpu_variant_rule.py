"""The stage kernel a context takes without the autotuner, where the choice
between staging paths, tiles and register budgets matters, and that the
kernels which are otherwise reached only by request agree with the others.

Bars, derived before the first run: the kernels compared differ in the
compiler's contractions of multiply-adds only.  FP64: 1e-14 relative L2, as
tests/test_gpu_dma_even.py.  FP32 storage: each of the two steps rounds the
stored state once (6e-8), so values agree but for flips of that rounding in a
part of the points: 1e-7, as tests/test_gpu_dma.py."""
import numpy as np
import pytest

from common import FIELDS, rel_l2, smooth_random_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import cosmograph_amd as cg
    cg.load_library()
    return cg


def context(gpu, prec, order, ko, lapse, shape, **kw):
    g = gpu.BSSN(gpu.GpuParams(n=shape, order=order, precision=prec, ko_coeff=ko, lapse=lapse, **kw))
    st = smooth_random_state(shape, seed=order, with_alpha=lapse != "Static")
    for f in FIELDS:
        g.upload(f + "_p", st[f])
    g.upload("DIFFD_a", st["DIFFD"])
    g.frw_set(0.0, -3.0)
    g.frw_add_fluid(3.0 / (8.0 * np.pi), 0.0)
    return g


PICKS = [
    # order 8 in split precision: LDS-DMA, with the tile of either halo
    ("fp32_split", 8, 0.0, "Static", (32, 32, 32), (4, 4, 16), True), ("fp32_split", 8, 0.0, "Harmonic", (32, 32, 48), (4, 4, 16), True),
    ("fp32_split", 8, 0.05, "Static", (32, 32, 32), (8, 8, 8), True), ("fp32_split", 8, 0.05, "Harmonic", (32, 24, 40), (8, 8, 8), True),
    # ... and where rows are no whole 16-byte groups
    ("fp32_split", 8, 0.0, "Harmonic", (31, 32, 33), (4, 8, 8), False), ("fp32_split", 8, 0.05, "Harmonic", (63, 64, 65), (8, 8, 8), False),
    # few tiles: a CU to each, so a tile of 512 points loses, and a round more or less decides
    ("fp64", 8, 0.0, "Static", (24, 24, 24), (4, 4, 16), True), ("fp64", 8, 0.0, "Harmonic", (40, 40, 39), (4, 8, 8), False),
    ("fp64", 8, 0.05, "Static", (30, 32, 25), (4, 8, 8), False), ("fp64", 8, 0.05, "Harmonic", (63, 64, 65), (8, 8, 8), False),
    ("fp64", 8, 0.05, "Static", (32, 32, 32), (8, 8, 8), True), ("fp64", 4, 0.0, "Static", (43, 47, 52), (4, 8, 8), True),
    ("fp64", 8, 0.0, "Static", (34, 42, 43), (8, 8, 8), False), ("fp32_split", 4, 0.0, "Harmonic", (59, 51, 56), (4, 4, 16), True),
    # ... and corner waves of 8 points: 2 rows of 4 in the 4x4x16 tile, 3 rows of 4 are full speed
    ("fp64", 4, 0.0, "Static", (20, 22, 20), (4, 8, 8), True), ("fp64", 4, 0.0, "Static", (20, 23, 20), (4, 4, 16), True),
    # order 2: the register budget of several waves outweighs some padding
    ("fp64", 2, 0.0, "Harmonic", (23, 24, 97), (4, 4, 16), False), ("fp32_split", 2, 0.0, "Static", (23, 24, 97), (4, 4, 16), False),
    # four-byte fields by registers, order 4: the kernel for four waves spills with a live lapse
    ("fp32_fix", 4, 0.0, "Harmonic", (31, 32, 61), (4, 8, 8), False), ("fp32_fix", 4, 0.0, "Static", (31, 32, 61), (4, 4, 16), False),
    ("fp32_all", 4, 0.0, "Harmonic", (31, 32, 61), (4, 8, 8), False), ("fp32_all", 4, 0.0, "Static", (31, 32, 61), (4, 4, 16), False),
    ("fp32_fix", 6, 0.0, "Harmonic", (31, 32, 61), (4, 4, 16), False), ("fp32_fix", 4, 0.0, "Harmonic", (32, 32, 64), (4, 4, 16), True),
]


@pytest.mark.parametrize("prec,order,ko,lapse,shape,tile,dma", PICKS)
def test_default(gpu, prec, order, ko, lapse, shape, tile, dma):
    g = context(gpu, prec, order, ko, lapse, shape)
    info = g.kernel_info()
    assert info["tile"] == tile, info
    g.set_dma(False)
    assert (context(gpu, prec, order, ko, lapse, shape, tile=tile).kernel_info() == info)
    assert (g.kernel_info() != info) == dma


def agree(a, b, tol):
    for f in FIELDS:
        assert rel_l2(a[f], b[f]) <= tol, (f, rel_l2(a[f], b[f]))


@pytest.mark.parametrize("prec", ["fp32_split", "fp64"])
@pytest.mark.parametrize("ko,shape", [(0.0, (17, 13, 32)), (0.0, (12, 20, 24)), (0.05, (18, 17, 24)), (0.05, (24, 16, 36))])
def test_order_8_staging(gpu, prec, ko, shape):
    print(f"case order 8 staging {prec} ko {ko} {shape}", flush=True)
    out, info = [], []
    for dma in (True, False):
        g = context(gpu, prec, 8, ko, "Harmonic", shape)
        g.set_dma(dma)
        g.step(2)
        out.append({f: g.download(f + "_p") for f in FIELDS})
        info.append(g.kernel_info())
    assert info[0] != info[1]  # the DMA kernel ran
    agree(out[0], out[1], 1e-14 if prec == "fp64" else 1e-7)


@pytest.mark.parametrize("prec", ["fp32_fix", "fp32_all"])
@pytest.mark.parametrize("order", [4, 6])
def test_register_staged_live_lapse(gpu, prec, order):
    """The 4x4x16 kernel of the four-byte modes by register staging with a live
    lapse (odd nz) against the 4x8x8 one."""
    print(f"case register staged live lapse {prec} order {order}", flush=True)
    out = []
    for tile in ((4, 4, 16), (4, 8, 8)):
        g = context(gpu, prec, order, 0.0, "Harmonic", (18, 13, 23), tile=tile)
        assert g.kernel_info()["tile"] == tile
        g.step(2)
        out.append({f: g.download(f + "_p") for f in FIELDS})
    agree(out[0], out[1], 1e-7)
