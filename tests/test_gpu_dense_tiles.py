"""density() and integrate() with particles crowded into few tiles: the tile's work is cut into pieces
of 4096 entries (N_p / 512 above 2 M particles), two pieces at least, shared out to many blocks.

Counts at the edges of the pieces (one entry below and above 2 and 3 of them), own and halo entries
each alone and together, more crowded halo lists than there are accumulators, one tile and eight in all, and
counts above 2^21.  Bars as for the tiles in general: a density cell is summed in float64 and rounded
once (2^-24 relative, 1e-7 asserted); a gradient is eight float32 products and sums, within 12 2^-24
times twice the largest |phi|, velocities and positions one float32 rounding on top.

A call's time follows its particle count, not how they are spread: without the pieces the crowded
calls below took 10 to 23 times the time of the spread one."""
import ctypes as C
import time

import numpy as np
import pytest

import pm_oracle as O
from helpers import periodic_diff

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24
PER = 4096


def _crowd(rng, count, lo, hi):
    """`count` positions in the box lo .. hi (cells)"""
    return rng.uniform(lo, hi, (count, 3)).T


def _case(name):
    rng = np.random.default_rng(len(name))
    if name.startswith("own"):                    # tile (1, 1, 1) of 16^3 on 96^3, away from its faces
        n, counts = 96, {"own-": 2 * PER - 1, "own": 2 * PER, "own+": 3 * PER - 1, "own++": 3 * PER}
        parts = [_crowd(rng, counts[name], 18, 30)]
    elif name.startswith("halo"):                 # on the upper x face of tile (0, 1, 1): halo of (1, 1, 1)
        n, counts = 96, {"halo-": 2 * PER - 1, "halo": 2 * PER, "halo+": 5 * PER + 1}
        m = counts[name]
        parts = [_crowd(rng, m, 18, 30)]
        parts[0][0] = 15 + rng.uniform(0.1, 0.9, m)
    elif name == "both":                          # a clump around a corner of eight tiles
        n, parts = 160, [np.mod(rng.normal(32, 1.5, (3, 200000)), 160)]
    elif name == "edge":                          # the same across the box's corner, in 8^3 tiles
        n, parts = 168, [np.mod(rng.normal(0, 1.5, (3, 200000)), 168)]
    elif name == "few tiles":
        n, parts = 16, [rng.uniform(0, 16, (3, 100000))]
    elif name == "one tile":
        n, parts = 8, [rng.uniform(0, 8, (3, 70001))]
    elif name == "corners":                       # every halo list of 729 tiles crowded, no own list is
        n, m = 72, 2880
        t = 8 * np.stack(np.meshgrid(*[np.arange(9)] * 3, indexing="ij")).reshape(3, 729, 1) + 7
        parts = [(t + rng.uniform(0, 1, (3, 729, m))).reshape(3, -1)]
    elif name == "large":
        n, parts = 176, [np.mod(rng.normal(40, 2.0, (3, 1 << 21)), 176), rng.uniform(0, 176, (3, 12345))]
    rest = 1 << 16
    parts.append(rng.uniform(0, n, (3, rest)))
    x = np.concatenate(parts, axis=1)
    x = x[:, rng.permutation(x.shape[1])].astype(np.float32)
    x[x >= n] = 0.0
    return n, x


CASES = ["own-", "own", "own+", "own++", "halo-", "halo", "halo+", "both", "edge", "one tile",
         "few tiles", "corners", "large"]


@pytest.mark.parametrize("name", CASES)
def test_density(name):
    from pmgpu import ops
    n, x = _case(name)
    got = ops.density(x, 7.3, n).astype(np.float64)
    want = O.density(x, 7.3, n)
    err = np.abs(got - want)
    print(f"{name}: n={n} n_p={x.shape[1]} max relative error {np.max(err / np.maximum(want, 1e-30)):.2e}")
    assert np.all(err <= 1e-7 * want + 1e-30)


@pytest.mark.parametrize("name", ["both", "edge", "large"])
def test_integrate(name):
    from pmgpu import ops
    n, x = _case(name)
    reps = max(1, -(-(1 << 19) // x.shape[1]))    # the tiled push starts at 2^19 particles
    x = np.ascontiguousarray(np.tile(x, reps))
    rng = np.random.default_rng(n)
    v = rng.normal(0, 0.3, x.shape).astype(np.float32)
    phi = rng.normal(0, 1, (n, n, n)).astype(np.float32)
    a, fa1, da = 0.3, 0.6, 0.05
    xr, vr = O.integrate(x, v, a, fa1, da, phi, n)
    ops.integrate(x, v, a, fa1, da, phi, n)
    vbar = da * fa1 * 12 * EPS * 2 * float(np.abs(phi).max()) + EPS * np.abs(vr)
    ev, ex = np.abs(v - vr), np.abs(periodic_diff(x, xr, n))
    print(f"{name}: velocity error {np.max(ev / vbar):.2f} of its bar, position {ex.max():.2e}")
    assert np.all(ev <= vbar)
    assert np.all(ex <= n * EPS + da * fa1 / (a + da) ** 2 * vbar)


def _times(n, x):
    """best times of one density and one integrate call on device arrays, us"""
    from pmgpu import _lib
    from pmgpu.device import DeviceArray
    n_p = x.shape[1]
    dx, dv = DeviceArray.from_numpy(x), DeviceArray.zeros(x.shape, np.float32)
    phi, rho = DeviceArray.zeros((n, n, n), np.float32), DeviceArray.zeros((n, n, n), np.float32)
    calls = [lambda: _lib.call("pm_density", dx.ptr, n_p, n, 1.0, rho.ptr),
             lambda: _lib.call("pm_integrate", dx.ptr, dv.ptr, n_p, n, C.c_double(0.5), 0.6, 0.0, phi.ptr)]
    out = []
    for f in calls:
        f()
        t = []
        for _ in range(8):
            t0 = time.perf_counter()
            f()
            t.append(time.perf_counter() - t0)
        out.append(1e6 * min(t))
    return out


def _uniform(n, n_p, seed=0):
    return np.random.default_rng(seed).uniform(0, n, (3, n_p)).astype(np.float32) % np.float32(n)


def _crowded(n, n_p, at, seed=0):
    """every other particle in one clump around `at` (cells) along each axis"""
    rng = np.random.default_rng(seed)
    x = rng.uniform(0, n, (3, n_p))
    x[:, ::2] = rng.normal(at, 1.0, x[:, ::2].shape)
    return np.mod(x, n).astype(np.float32) % np.float32(n)


def test_time_does_not_grow_with_crowding():
    n_p = 1 << 21
    spread = _times(256, _uniform(256, n_p))
    crowded = {"clump": _times(256, _crowded(256, n_p, 100.0)), "one tile": _times(16, _uniform(16, n_p))}
    print(f"spread: density {spread[0]:.0f} us, integrate {spread[1]:.0f} us")
    for name, t in crowded.items():
        print(f"{name}: density {t[0]:.0f} us, integrate {t[1]:.0f} us")
        assert t[0] < 3 * spread[0] and t[1] < 3 * spread[1]
