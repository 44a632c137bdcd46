"""The FP64 z pass that keeps its columns in registers (N = 256 and 512) against the LDS pass, which
the same sim runs with half the columns per block, in the three k-space forms: the analytic Green's
function, the CIC-deconvolved one and a caller's float32 grid (one that is not mirror-symmetric, so
the pass takes its Hermitian part).  Same bar as for any two pencil shapes at FP64: 1e-13 norm-wise.
"""
import numpy as np
import pytest

from helpers import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 512])
@pytest.mark.parametrize("form", ["plain", "deconvolve", "grid"])
def test_register_z_pass_against_the_lds_pass(n, form):
    from pmgpu.device import DeviceArray
    from pmgpu.sim import PMSim
    rng = np.random.default_rng(n)
    x = rng.uniform(0, n, (3, 64 ** 3))
    v = np.zeros_like(x)
    g = DeviceArray.from_numpy(rng.uniform(0.1, 2.0, (n, n, n)).astype(np.float32)) if form == "grid" else None
    phi = []
    for z in (0, 4):
        sim = PMSim(n, 64, 64, cic_deconvolve=form == "deconvolve", deterministic=True, omega_m0=0.3,
                    omega_lambda0=0.7, h0=0.7)
        sim.set_pencils(0, z, 0)
        if g is not None:
            sim.set_green(g)
        sim.set_state(x, v)
        sim.step(0.25, 1e-3)
        phi.append(sim.potential(np.float64))
        sim.close()
    e = rel(phi[0], phi[1])
    print(f"N={n} {form}: register against LDS z pass {e:.1e}")
    assert e < 1e-13
