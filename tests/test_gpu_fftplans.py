"""The FFT plans kept between calls: the same answers from a kept plan, from
plans of several grids in turn (more of them than the pool keeps), and from
contexts used by several threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spectrum(cg, shape, seed):
    g = cg.BSSN(cg.GpuParams(n=shape, order=4))
    x = np.random.default_rng(seed).standard_normal(shape)
    g.upload("DIFFphi_p", x)
    return g, x


def reference(x):
    nx, ny, nz = x.shape
    k = [np.fft.fftfreq(n, d=1.0 / n) for n in (nx, ny)] + [np.arange(nz // 2 + 1.0)]
    kx, ky, kz = np.meshgrid(*k, indexing="ij")
    w = np.where((kz > 0) & (kz < nz // 2), 2.0, 1.0)
    b = np.sqrt(kx * kx + ky * ky + kz * kz).astype(int)
    nb = int(np.sqrt(float(nx * nx + ny * ny + nz * nz)) / 2.0) + 1
    f = np.bincount(b.ravel(), (w * np.abs(np.fft.rfftn(x)) ** 2).ravel(), nb)[:nb]
    c = np.bincount(b.ravel(), w.ravel(), nb)[:nb]
    return np.where(c > 0, f / np.maximum(c, 1), 0.0)


def close(got, x):
    np.testing.assert_allclose(got, reference(x), rtol=1e-12, atol=0)


def test_many_grids_in_turn():
    import cosmograph_amd as cg
    shapes = [(12 + 2 * q, 16, 20 + 2 * q) for q in range(11)]
    kept = [spectrum(cg, s, 3 + q) for q, s in enumerate(shapes)]
    for _ in range(2):
        for g, x in kept:
            close(g.power_spectrum("DIFFphi_a"), x)


def test_threads():
    import cosmograph_amd as cg
    shapes = [(16, 16, 16), (16, 16, 16), (24, 16, 16), (16, 16, 16)]
    bad = []

    def work(q):
        try:
            g, x = spectrum(cg, shapes[q], 40 + q)
            for _ in range(8):
                close(g.power_spectrum("DIFFphi_a"), x)
        except BaseException as e:  # noqa: BLE001
            bad.append(repr(e))
    ts = [threading.Thread(target=work, args=(q,)) for q in range(len(shapes))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_plan_outlives_its_context():
    import cosmograph_amd as cg
    g, x = spectrum(cg, (16, 18, 20), 1)
    a = g.power_spectrum("DIFFphi_a")
    del g
    g, x = spectrum(cg, (16, 18, 20), 2)
    close(g.power_spectrum("DIFFphi_a"), x)
    assert not np.array_equal(a, g.power_spectrum("DIFFphi_a"))
