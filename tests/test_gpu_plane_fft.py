"""The plane passes (x and y of a z plane in one block) against the separate x and y passes, which the
same sim runs when a y pencil shape is chosen: the plane passes run the same butterflies, so a step
with the order-independent deposit gives the same bits.  Also the x margins they write for 32-wide
tiles, and the stateless solve at the smallest sizes against the oracle (FP64 FFT, one float32
rounding: 1e-6 norm-wise)."""
import numpy as np
import pytest

import pm_oracle as O
from helpers import rel

pytestmark = pytest.mark.gpu

KW = dict(omega_m0=0.3, omega_lambda0=0.7, omega_k0=0.0, h0=0.7)


@pytest.mark.parametrize("n,prec,tiles", [(64, 32, (0, 0, 0)), (64, 32, (32, 8, 8)), (96, 32, (0, 0, 0)),
                                          (128, 32, (0, 0, 0)), (192, 32, (0, 0, 0)), (192, 32, (32, 8, 8)),
                                          (64, 64, (0, 0, 0)), (96, 64, (0, 0, 0)), (128, 64, (0, 0, 0))])
def test_plane_passes_give_the_bits_of_separate_passes(n, prec, tiles):
    from pmgpu.sim import PMSim
    rng = np.random.default_rng(n)
    side = 32
    x = rng.uniform(0, n, (3, side ** 3)).astype(np.float32)
    v = rng.normal(0, 1, (3, side ** 3)).astype(np.float32)
    out = []
    for alt in (False, True):
        s = PMSim(n, side, prec, deterministic=True, **KW)
        s.set_tiles(*tiles)
        if alt:
            w = s.pencils()[0] // 2
            s.set_pencils(w, 0, w)
        s.set_state(x, v)
        s.run(0.3, 0.01, 9)
        out.append((s.potential(np.float64), *s.get_state(np.float64)))
        s.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("n", [8, 16, 32, 48, 64, 128])
def test_small_poisson_solves(n):
    from pmgpu import ops
    rng = np.random.default_rng(n)
    rho = rng.uniform(0, 2, (n, n, n)).astype(np.float32)
    g = O.fourier_grid(n).astype(np.float32)
    want = O.potential(rho.astype(np.float64), g.astype(np.float64), 0.4, 0.3)
    assert rel(ops.potential(rho, g, 0.4, 0.3), want) < 1e-6
    k = ops.density_k(rho)
    assert rel(k, O.density_k(rho.astype(np.float64))) < 1e-12
    assert rel(ops.potential_real(ops.potential_k(k, g, 0.4, 0.3)), want) < 1e-6
