"""The default tile shape of every grid size and both forms of the tile scatter (one wavefront per
tile from 16384 tiles on, four below) against 8^3 tiles, which take the particle-parallel scatter:
with the order-independent deposit the shape changes no bit of a run.  Clustered particles (dense
tiles of several batches) that cross many tile faces, some by more than one tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KW = dict(omega_m0=0.3, omega_lambda0=0.7, omega_k0=0.0, h0=0.7)
DEFAULTS = {8: (8, 8, 8), 16: (8, 8, 8), 32: (8, 8, 8), 48: (8, 8, 8), 64: (8, 8, 8), 96: (16, 16, 8),
            128: (16, 16, 8), 192: (16, 16, 8), 256: (32, 8, 8), 384: (32, 8, 8)}


def _state(n, side, seed):
    rng = np.random.default_rng(seed)
    m = side ** 3
    x = rng.uniform(0, n, (3, m))
    x[:, : m // 2] = np.mod(rng.normal(n * 0.99, n / 24, (3, m // 2)), n)
    v = rng.normal(0, 40.0, (3, m))
    return x.astype(np.float32) % np.float32(n), v.astype(np.float32)


@pytest.mark.parametrize("n,prec", [(n, 32) for n in DEFAULTS] + [(64, 64), (96, 64), (256, 64)])
def test_default_tiles_give_the_bits_of_8_cubed(n, prec):
    from pmgpu.sim import PMSim
    side = min(max(n // 2, 4), 96)
    x, v = _state(n, side, n)
    out = []
    for tiles in ((0, 0, 0), (8, 8, 8)):
        s = PMSim(n, side, prec, deterministic=True, **KW)
        assert s.tiles() == DEFAULTS[n]
        s.set_tiles(*tiles)
        s.set_state(x, v)
        s.run(0.5, 0.01, 11)
        out.append((s.density(np.float64), *s.get_state(np.float64)))
        s.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


def test_member_keeps_the_ensemble_shape():
    from pmgpu.ensemble import PMEnsemble
    from pmgpu.sim import PMSim
    from pmgpu.ensemble import ensemble_tiles
    for n in (48, 64, 128, 256):
        s = PMSim(n, 32, 32, **KW)
        s.set_tiles(16, 16, 16)
        ens = PMEnsemble([s])
        assert s.tiles() == ensemble_tiles(n)
        for tiles in ((0, 0, 0), (16, 16, 16)):      # both leave a member where it is
            s.set_tiles(*tiles)
            x, v = _state(n, 32, 1)
            s.set_state(x, v)
            ens.run([0.5], [0.001], 2)
            assert s.tiles() == ensemble_tiles(n)
        with pytest.raises(RuntimeError):
            s.set_tiles(8, 8, 8)
        ens.close()
