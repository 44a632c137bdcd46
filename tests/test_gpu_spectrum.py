"""The shell sums of the power spectrum, mode by mode."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec,bins", [(8, 32, 4), (8, 64, 20), (48, 64, 1), (64, 32, 32), (96, 64, 200), (128, 64, 64)])
def test_shell_sums_over_every_mode(n, prec, bins):
    # power_spectrum against the same sums over the full DFT in numpy: mirrored modes, the planes
    # with and without a mirror image, bins beyond the last mode (empty) and before it (left out).
    # The counts are whole numbers; k sums exact roots in float64 (1e-13); P(k) carries the FFT's
    # rounding in the sim's precision (1e-5 FP32, 1e-11 FP64 per shell)
    from pmgpu.sim import PMSim
    s = PMSim(n, 8, prec)
    rng = np.random.default_rng(n)
    x = rng.uniform(0, n, (3, 512))
    s.set_state(x, np.zeros_like(x))
    s.deposit()
    rho = s.density(np.float64)
    k, pk, cnt = s.power_spectrum(100.0, bins)
    s.close()
    f = np.abs(np.fft.fftn(rho / rho.mean() - 1)) ** 2
    m = np.fft.fftfreq(n, 1 / n)
    r = np.sqrt(m[:, None, None] ** 2 + m[None, :, None] ** 2 + m[None, None, :] ** 2)
    b = np.floor(r + 0.5).astype(int).ravel()
    size = max(b.max(), bins) + 1
    c = np.bincount(b, minlength=size)[1:bins + 1]
    assert np.array_equal(cnt, c)
    ok = c > 0
    order = np.argsort(b, kind="stable")
    edges = np.searchsorted(b[order], np.arange(1, bins + 2))
    kr = np.array([math.fsum(r.ravel()[order[i:j]]) for i, j in zip(edges[:-1], edges[1:])])[ok] / c[ok]
    pr = np.bincount(b, f.ravel(), size)[1:bins + 1][ok] / c[ok] * 100.0 ** 3 / float(n) ** 6
    assert np.allclose(k[ok], kr * 2 * np.pi / 100.0, rtol=1e-13, atol=0)
    assert np.all(np.abs(pk[ok] - pr) <= (1e-5 if prec == 32 else 1e-11) * pr.max())
    assert np.all(pk[~ok] == 0)
