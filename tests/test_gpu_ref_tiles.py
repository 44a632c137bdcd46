"""The tiled density() and integrate() of the reference-layout entry points against the oracle.

Sizes at the edges of the tiles (8^3 and 16^3, one tile per axis, an odd number of them), of the three
forms of the binning (up to 8192 tile keys, up to 36864 from 2^21 particles on, above), of the
particle mapping (cubes of odd sides, counts that are no cube) and of the rule that takes them (the
smallest counts; a grid no tile divides), in lattice and in random order, with particles on tile faces and on the box's edge.

Bars: the density of a cell is summed in float64 and rounded once (2^-24 relative, 1e-7 asserted).
The gradient is eight float32 products of weights (2^-24 each) and differences of float32
potentials (2^-24 |phi| each), summed in float32: within 12 2^-24 times twice the largest |phi|;
velocities and positions add one float32 rounding each.
"""
import numpy as np
import pytest

import pm_oracle as O
from helpers import periodic_diff

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _positions(n, n_p, order, seed):
    rng = np.random.default_rng(seed)
    side = int(round(n_p ** (1 / 3)))
    if order == "lattice" and side ** 3 == n_p:
        x = O.lattice_q(side, n, np.float64) + rng.normal(0, 0.4, (3, n_p))
        x = np.mod(x, n).astype(np.float32)
    else:  # two thirds spread over the box, the rest in one clump, in random order
        x = rng.uniform(0, n, (3, n_p))
        m = n_p // 3
        x[:, :m] = np.mod(rng.normal(n - 0.3, 1.0, (3, m)), n)
        x = x[:, rng.permutation(n_p)].astype(np.float32)
    x[x >= n] = 0.0
    x[:, 0] = 0.0
    x[:, 1] = n                                  # stored as n: wraps to 0
    x[:, 2] = np.nextafter(np.float32(n), np.float32(0))
    x[:, 3] = min(16, n - 1)                     # a tile face
    x[:, 4] = np.nextafter(np.float32(min(16, n - 1)), np.float32(0))
    return x


DENSITY = [(8, 65536, "random"), (16, 65536, "random"), (24, 65537, "random"), (20, 65537, "random"),
           (48, 41 ** 3, "lattice"), (96, 51 ** 3, "lattice"), (128, 64 ** 3, "lattice"),
           (256, 65536, "random"), (264, 80 ** 3, "lattice"), (272, 300001, "random"), (288, 100 ** 3, "lattice"),
           (272, 2 ** 21, "random"), (416, 2 ** 21 + 1, "random"), (432, 2 ** 21 + 1, "random")]


@pytest.mark.parametrize("n,n_p,order", DENSITY)
def test_density(n, n_p, order):
    from pmgpu import ops
    x = _positions(n, n_p, order, seed=n)
    got = ops.density(x, 7.3, n).astype(np.float64)
    want = O.density(x, 7.3, n)
    err = np.abs(got - want)
    print(f"n={n} n_p={n_p}: max relative error {np.max(err / np.maximum(want, 1e-30)):.2e}")
    # (a grid no tile divides keeps float32 sums: one rounding per contribution)
    assert np.all(err <= (1e-7 if n % 8 == 0 else 1e-5) * want + 1e-30)


PUSH = [(16, 1 << 19, "random"), (24, (1 << 19) + 1, "random"), (96, 81 ** 3, "lattice"),
        (160, 81 ** 3, "random"), (168, 83 ** 3, "lattice"), (336, 700001, "random"), (352, 81 ** 3, "lattice"),
        (336, 2 ** 21, "random"), (416, 2 ** 21 + 1, "random")]


@pytest.mark.parametrize("n,n_p,order", PUSH)
def test_integrate(n, n_p, order):
    from pmgpu import ops
    x = _positions(n, n_p, order, seed=n)
    rng = np.random.default_rng(n + 1)
    v = rng.normal(0, 0.3, (3, n_p)).astype(np.float32)
    phi = rng.normal(0, 1, (n, n, n)).astype(np.float32)
    a, fa1, da = 0.3, 0.6, 0.05
    xr, vr = O.integrate(x, v, a, fa1, da, phi, n)
    xg, vg = x.copy(), v.copy()
    ops.integrate(xg, vg, a, fa1, da, phi, n)
    gmax = 12 * EPS * 2 * float(np.abs(phi).max())
    vbar = da * fa1 * gmax + EPS * np.abs(vr)
    ev = np.abs(vg - vr)
    ex = np.abs(periodic_diff(xg, xr, n))
    print(f"n={n} n_p={n_p}: velocity error {np.max(ev / vbar):.2f} of its bar, position {ex.max():.2e}")
    assert np.all(ev <= vbar)
    assert np.all(ex <= n * EPS + da * fa1 / (a + da) ** 2 * vbar)
