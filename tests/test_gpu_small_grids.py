"""density() and integrate() with many particles on small grids take no longer through the tiles than
without: the same call on a slightly different grid that no tile divides is the measure."""
import pytest

from test_gpu_dense_tiles import _times, _uniform

pytestmark = pytest.mark.gpu


def test_integrate_small_grid():
    n_p = 1 << 21
    tiled, plain = _times(64, _uniform(64, n_p))[1], _times(60, _uniform(60, n_p))[1]
    print(f"integrate: 64^3 {tiled:.0f} us, 60^3 {plain:.0f} us")
    assert tiled < 1.35 * plain


def test_density_small_grid():
    n_p = 57 ** 3
    tiled, plain = _times(32, _uniform(32, n_p))[0], _times(36, _uniform(36, n_p))[0]
    print(f"density: 32^3 {tiled:.0f} us, 36^3 {plain:.0f} us")
    assert tiled < 1.35 * plain
