"""Tile shapes of a sim that is a member of an ensemble: its own shape can be asked for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KW = dict(omega_m0=0.3, omega_lambda0=0.7, omega_k0=0.0, h0=0.7)


@pytest.mark.parametrize("n", [64, 128])
def test_a_member_accepts_its_own_shape(n):
    from pmgpu.ensemble import PMEnsemble, ensemble_tiles
    from pmgpu.sim import PMSim
    s = PMSim(n, 32, 32, **KW)
    ens = PMEnsemble([s])
    x = np.random.default_rng(n).uniform(0, n, (3, 32 ** 3)).astype(np.float32) % np.float32(n)
    s.set_state(x, np.zeros_like(x))
    for tiles in (ensemble_tiles(n), s.tiles()):
        s.set_tiles(*tiles)
        assert s.tiles() == ensemble_tiles(n)
    other = (16, 16, 8) if n >= 128 else (32, 8, 8)
    with pytest.raises(RuntimeError):
        s.set_tiles(*other)
    assert s.tiles() == ensemble_tiles(n)
    ens.run([0.5], [0.001], 2)
    ens.close()
    s.close()
