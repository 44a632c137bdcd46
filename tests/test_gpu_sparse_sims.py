"""Sims of few particles (more than 16 cells each): their default tiles on small grids are 16^3, and a step takes no longer in them than in 16^3 asked for.  With the
order-independent deposit neither the shape nor the form of the scatter (one wavefront for tiles of few
particles) changes a bit of a run, alone or in an ensemble."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KW = dict(omega_m0=0.3, omega_lambda0=0.7, omega_k0=0.0, h0=0.7)


def _state(n, side):
    rng = np.random.default_rng(n + side)
    q = np.arange(side) * (n / side) + 0.5
    x = np.stack([g.ravel() for g in np.meshgrid(q, q, q, indexing="ij")]) + rng.normal(0, 2.0, (3, side ** 3))
    v = rng.normal(0, 20.0, (3, side ** 3))
    return np.mod(x, n).astype(np.float32) % np.float32(n), v.astype(np.float32)


@pytest.mark.parametrize("n,side,prec,tiles", [(32, 4, 32, (16, 16, 16)), (64, 16, 32, (16, 16, 16)), (64, 32, 32, (8, 8, 8)),
                                               (64, 8, 64, (16, 16, 16)), (192, 64, 32, (16, 16, 8)),
                                               (192, 96, 32, (16, 16, 8)), (256, 64, 32, (32, 8, 8))])
def test_shape_and_bits(n, side, prec, tiles):
    from pmgpu.sim import PMSim
    x, v = _state(n, side)
    out = []
    for shape in ((0, 0, 0), (8, 8, 8)):
        s = PMSim(n, side, prec, deterministic=True, **KW)
        assert s.tiles() == tiles
        s.set_tiles(*shape)
        assert s.tiles() == (tiles if shape == (0, 0, 0) else shape)
        s.set_state(x, v)
        s.run(0.5, 0.01, 11)
        out.append((s.density(np.float64), *s.get_state(np.float64)))
        s.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("grids", [((192, 48), (128, 32), (64, 16)), ((256, 128), (96, 48), (192, 96), (48, 24))])
def test_members_keep_the_bits_of_lone_runs_in_their_tiles(grids):
    from pmgpu.ensemble import PMEnsemble
    from pmgpu.sim import PMSim
    sims, lone = [], []
    for n, side in grids:
        x, v = _state(n, side)
        for group in (sims, lone):
            s = PMSim(n, side, 32, deterministic=True, **KW)
            s.set_state(x, v)
            group.append(s)
    ens = PMEnsemble(sims)
    ens.run([0.5] * len(sims), [0.01] * len(sims), 9)
    for a, b in zip(sims, lone):
        b.set_tiles(*a.tiles())
        b.run(0.5, 0.01, 9)
        for p, q in zip(a.get_state(np.float64), b.get_state(np.float64)):
            assert np.array_equal(p, q)
    ens.close()
    for s in sims + lone:
        s.close()


def test_step_of_few_particles():
    from pmgpu.sim import PMSim
    n, side = 64, 8
    x, v = _state(n, side)
    s = PMSim(n, side, 32, **KW)

    def step(shape):
        s.set_tiles(*shape)
        s.set_state(x, 0 * v)
        t = []
        for _ in range(9):
            t0 = time.perf_counter()
            s.run(0.5, 1e-9, 64)
            t.append((time.perf_counter() - t0) / 64 * 1e6)
        return sorted(t)[4]

    default, cube = step((0, 0, 0)), step((16, 16, 16))
    print(f"step of {side}^3 particles on {n}^3: default tiles {default:.1f} us, 16^3 {cube:.1f}")
    assert default < 1.3 * cube
    s.close()
