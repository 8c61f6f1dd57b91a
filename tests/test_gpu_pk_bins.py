"""Binned power spectrum at the edges of its wave sums: one bin, more bins
than a row has runs, rows longer and shorter than a wave, the full spectrum of
a side without a register plan, and a change of the bin count on one context."""
import numpy as np
import pytest

import simfast21_amd as sf

pytestmark = pytest.mark.gpu


def reference(field, side, nbins):
    """tools/power3d.c's normalisation on numpy's FP64 transform."""
    n = field.shape[0]
    spec = np.fft.rfftn(field.astype(np.float64))
    f = np.rint(np.fft.fftfreq(n) * n)
    m = f[:, None, None] ** 2 + f[None, :, None] ** 2 + np.arange(n // 2 + 1)[None, None, :] ** 2
    k = np.sqrt(m)
    b = np.minimum(np.floor((k - 1) / ((n // 2 - 1) / nbins)), nbins - 1).astype(int)
    keep = (k >= 1) & (k <= n // 2)
    count = np.bincount(b[keep], minlength=nbins).astype(float)
    power = np.bincount(b[keep], (np.abs(spec) ** 2)[keep], nbins)
    kk = np.bincount(b[keep], k[keep], nbins)
    some = np.maximum(count, 1)
    return power / some * (side / n) ** 3 / n ** 3, kk / some * 2 * np.pi / side, count


@pytest.mark.parametrize("n", [64, 80, 128, 192])
def test_bins(torch_cuda, n):
    torch = torch_cuda
    side = 1.5 * n
    field = np.random.default_rng(n).standard_normal((n, n, n)).astype(np.float32)
    dev = torch.from_numpy(field.ravel()).cuda()
    ctx = sf.HiiContext(n, side, [side / n], sf.INPUT_DIRECT, sf.PATH_FUSED, radius_batch=1)
    for nbins in (1, 64, 20):
        pk, km, ct = ctx.power_spectrum(dev, nbins)
        rp, rk, rc = reference(field, side, nbins)
        assert np.array_equal(ct, rc), (n, nbins)
        # FP32 transform: 2e-6 of the largest mode, doubled by the square and
        # averaged; the same bars as the oracle comparison of the spectrum
        assert np.all(np.abs(pk - rp) <= 2e-5 * rp), (n, nbins)
        assert np.all(np.abs(km - rk) <= 1e-6 * rk), (n, nbins)
        again = ctx.power_spectrum(dev, nbins)
        assert np.array_equal(again[1], km) and np.array_equal(again[2], ct)
    ctx.close()
