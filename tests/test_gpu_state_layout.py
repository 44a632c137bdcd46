"""State in and out of a resident sim, in every storage order a sim can be in: slot order (just set,
lattices of 4^3 blocks and others, sides at and off the edges of the 64-site runs) and tile order
(after steps, replayed graphs and ensemble runs).  With a zero time step every particle keeps its
position and velocity, so what comes out is what went in, each at its reference index: float64 sims
hold the displacement x - q to 2^-53 (positions within 1e-13 of a cell at N <= 192), float32 sims to
2^-24 of the largest displacement plus the float32 position's own rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 72


def _state(side, seed, dtype):
    rng = np.random.default_rng(seed)
    q = np.stack([g.reshape(-1) for g in np.meshgrid(*[np.arange(side) * (N / side) + 0.5] * 3, indexing="ij")])
    x = np.mod(q + rng.normal(0, 2.0, q.shape), N).astype(dtype)
    x[x >= N] = 0.0
    return x, rng.normal(0, 1.0, q.shape).astype(dtype)


def _check(got, want, prec):
    from helpers import periodic_diff
    (x, v), (x0, v0) = got, want
    assert np.array_equal(v, v0)
    bar = 1e-13 if prec == 64 else N * 2.0 ** -23
    assert np.abs(periodic_diff(x, x0, N)).max() <= bar


@pytest.mark.parametrize("side", [4, 5, 16, 20, 33, 34, 36, 80, 81, 84, 92])
@pytest.mark.parametrize("prec", [32, 64])
def test_state_comes_back_at_its_reference_index(side, prec):
    from pmgpu.sim import PMSim
    n = 48 if side < 20 else 96 if side < 80 else 192
    global N
    N = n
    dt = np.float32 if prec == 32 else np.float64
    x, v = _state(side, side, dt)
    for graph in (True, False):
        s = PMSim(n, side, prec, graph=graph, omega_m0=0.3, omega_lambda0=0.7, h0=0.7)
        s.set_state(x, v)
        _check(s.get_state(dt), (x, v), prec)         # slot order
        s.step(0.5, 0.0)
        _check(s.get_state(dt), (x, v), prec)         # tile order
        for steps in (9, 17, 16):                     # graph replays, with and without remainder
            s.set_state(x, v)
            s.run(0.5, 0.0, steps)
            _check(s.get_state(dt), (x, v), prec)
        s.close()


def test_state_after_ensemble_runs():
    from pmgpu.ensemble import PMEnsemble
    from pmgpu.sim import PMSim
    global N
    N = 96
    sims = [PMSim(96, p, 32, omega_m0=0.3, omega_lambda0=0.7, h0=0.7) for p in (32, 84)]
    states = [_state(p, 7, np.float32) for p in (32, 84)]
    ens = PMEnsemble(sims)
    for steps in (1, 64, 8):
        for s, (x, v) in zip(sims, states):
            s.set_state(x, v)
        ens.run([0.5] * 2, [0.0] * 2, steps)
        for s, (x, v) in zip(sims, states):
            _check(s.get_state(), (x, v), 32)
    ens.close()


def test_non_finite_values_are_counted_once_per_particle():
    from pmgpu.sim import PMSim
    global N
    N = 96
    for side in (20, 33, 84):
        x, v = _state(side, 3, np.float32)
        x[1, 17] = np.nan
        v[2, 17] = np.inf
        v[0, 40] = np.nan
        s = PMSim(96, side, 32)
        with pytest.raises(RuntimeError, match="2 non-finite"):
            s.set_state(x, v)
        s.close()
