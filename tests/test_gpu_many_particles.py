"""density() and integrate() of more particles than the kept scratch buffer has room for at 8 entries each
(33 M): the bins are sized to what they hold, no buffer is allocated and freed by each call.

A density adds up: all particles together against the sum of two halves, which take the ordinary path.
Cells are float64 sums rounded once (2^-24), so with the two halves' roundings and that of their sum
4 2^-24 of the cell."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _positions(n, n_p, seed):
    x = np.random.default_rng(seed).random((3, n_p), dtype=np.float32) * np.float32(n)
    x[x >= n] = 0
    return x


def _density(x, n):
    from pmgpu import ops
    return ops.density(np.ascontiguousarray(x), 1.5, n).astype(np.float64)


@pytest.mark.parametrize("n_p", [33_000_000, 40_000_001])
def test_density_adds_up(n_p):
    n, half = 256, n_p // 2
    x = _positions(n, n_p, n_p)
    both, parts = _density(x, n), _density(x[:, :half], n) + _density(x[:, half:], n)
    assert np.all(np.abs(both - parts) <= 4 * EPS * parts)
    assert abs(both.sum() / (1.5 * n_p) - 1) < 1e-7


def test_density_of_entries_that_do_not_fit():
    """every particle on a corner of eight tiles: 8 entries each, so the call runs without bins (float32
    sums: 2^-24 per contribution at most)"""
    n, n_p = 512, 40_000_000
    half = n_p // 2
    rng = np.random.default_rng(1)
    x = rng.random((3, n_p), dtype=np.float32) * np.float32(0.99)
    x += 16 * rng.integers(0, n // 16, (3, n_p), dtype=np.int16) + np.float32(15)
    both, parts = _density(x, n), _density(x[:, :half], n) + _density(x[:, half:], n)
    per_cell = 2 * n_p / (n // 16) ** 3
    assert np.all(np.abs(both - parts) <= per_cell * EPS * parts + 1e-6)
    assert abs(both.sum() / (1.5 * n_p) - 1) < 1e-4


def test_no_allocation_per_call():
    """calls in a loop: three times the particles, three times the time.  A loop that frees and allocates 32
    bytes a particle in each call outruns the driver's clearing of freed memory: once what was free at
    first is used up, after some 110 calls, it waits for it (57.6 ms a density call instead of 17.2)."""
    from pmgpu import _lib
    from pmgpu.device import DeviceArray
    n = 512
    phi, rho = DeviceArray.zeros((n, n, n), np.float32), DeviceArray.zeros((n, n, n), np.float32)

    def times(n_p):
        x, v = DeviceArray.from_numpy(_positions(n, n_p, 3)), DeviceArray.zeros((3, n_p), np.float32)
        out = []
        for f in (lambda: _lib.call("pm_density", x.ptr, n_p, n, 1.0, rho.ptr),
                  lambda: _lib.call("pm_integrate", x.ptr, v.ptr, n_p, n, 0.5, 0.6, 0.0, phi.ptr)):
            t = []
            for _ in range(200 if n_p > 50_000_000 else 20):
                t0 = time.perf_counter()
                f()
                t.append(time.perf_counter() - t0)
            out.append(1e3 * sorted(t[-12:])[6])
        return out

    few, many = times(30_000_001), times(100_000_001)
    print(f"30 M: density {few[0]:.1f} ms, integrate {few[1]:.1f}; 100 M: {many[0]:.1f} and {many[1]:.1f}")
    assert many[0] < 5 * few[0] and many[1] < 5 * few[1]
