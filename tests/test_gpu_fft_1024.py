"""The FP32 passes at N = 1024 (16 columns of 32 threads, real and imaginary parts exchanged in turn,
the spectrum moved into pages by the forward y pass and back by the inverse one) against the FP64 sim,
whose passes at that size go through LDS in the plain layout: potential of the same density.

Bar: 1e-5 norm-wise, as for every FP32 potential against float64 here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("deconvolve", [False, True])
def test_potential_at_1024(deconvolve):
    import ctypes as C

    import torch
    from pmgpu import _lib
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
        out = torch.empty((n,) * 3, dtype=torch.float32, device="cuda")
        _lib.call("pm_sim_get_potential", sim._h, C.c_void_p(out.data_ptr()), 4, 1)
        sim.close()
        phi.append(out)
    a, b = phi
    err, norm = 0.0, 0.0
    for z in range(0, n, 64):
        p, q = a[z:z + 64].double(), b[z:z + 64].double()
        err += float((p - q).square().sum())
        norm += float(q.square().sum())
    e = (err / norm) ** 0.5
    print(f"N=1024 deconvolve={deconvolve}: potential FP32 against FP64 {e:.1e}")
    assert e < 1e-5
