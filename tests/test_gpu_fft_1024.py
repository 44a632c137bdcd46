"""The FP32 passes at N = 1024 (16 columns of 32 threads, real and imaginary parts exchanged in turn,
the spectrum moved into pages by the forward y pass and back by the inverse one) against the FP64 sim,
whose passes at that size go through LDS in the plain layout: potential of the same density.

Bar: 1e-5 norm-wise, as for every FP32 potential against float64 here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("deconvolve", [False, True])
def test_potential_at_1024(deconvolve):
    from pmgpu.sim import PMSim
    n, side = 1024, 64
    rng = np.random.default_rng(5)
    x = rng.uniform(0, n, (3, side ** 3)).astype(np.float32)
    v = np.zeros_like(x)
    phi = []
    for prec in (32, 64):
        sim = PMSim(n, side, prec, cic_deconvolve=deconvolve, omega_m0=0.3, omega_lambda0=0.7, h0=0.7)
        sim.set_state(x, v)
        sim.step(0.25, 1e-3)
        phi.append(sim.potential(np.float32))
        sim.close()
    a, b = phi
    err, norm = 0.0, 0.0
    for z in range(0, n, 64):
        p, q = a[z:z + 64].astype(np.float64), b[z:z + 64].astype(np.float64)
        err += float(((p - q) ** 2).sum())
        norm += float((q ** 2).sum())
    e = (err / norm) ** 0.5
    print(f"N=1024 deconvolve={deconvolve}: potential FP32 against FP64 {e:.1e}")
    assert e < 1e-5
