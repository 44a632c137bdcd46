"""Binning of particles in no order on grids of many tiles (counters of every wavefront in device memory),
half of them in one tile or around the corner of eight: the crowd of a wavefront takes one place at its
tile's counter, however its lanes are mixed with others.

Bars as for the tiles: a density cell is summed in float64 and rounded once (1e-7 relative)."""
import numpy as np
import pytest

import pm_oracle as O
from test_gpu_dense_tiles import _crowded, _times, _uniform

pytestmark = pytest.mark.gpu

N, N_P = 384, 128 ** 3                  # 13824 tiles; a cube of particles, so never the wide LDS table


@pytest.mark.parametrize("at", [200.0, 192.0, 0.0])      # inside a tile, a corner of eight, the box's corner
def test_density_of_a_crowd(at):
    from pmgpu import ops
    x = _crowded(N, N_P, at)
    got = ops.density(x, 7.3, N).astype(np.float64)
    want = O.density(x, 7.3, N)
    assert np.all(np.abs(got - want) <= 1e-7 * want + 1e-30)


@pytest.mark.parametrize("at", [200.0, 192.0])
def test_crowds_do_not_queue(at):
    spread, crowded = _times(N, _uniform(N, N_P)), _times(N, _crowded(N, N_P, at))
    print(f"spread: {spread[0]:.0f} and {spread[1]:.0f} us, crowded at {at}: {crowded[0]:.0f} and {crowded[1]:.0f}")
    assert crowded[0] < 8 * spread[0] and crowded[1] < 4 * spread[1]
