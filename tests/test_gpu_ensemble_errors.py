"""A batched call that ends early (a member's scale factor would turn negative in a later part of the
call) keeps the steps it took: each member's state reads as after those steps, particle by particle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KW = dict(omega_m0=0.3, omega_lambda0=0.7, omega_k0=0.0, h0=0.7)
CHUNK = 1024  # steps whose scalars one call uploads together


def _member(n, side, x, v):
    from pmgpu.sim import PMSim
    s = PMSim(n, side, 32, deterministic=True, **KW)
    s.set_state(x, v)
    return s


# sizes around the line from which a state goes in and out in whole cache lines (2^19 particles)
@pytest.mark.parametrize("side", [40, 84])
def test_state_after_a_call_that_ends_early(side):
    from pmgpu.ensemble import PMEnsemble
    n, a0, da = 32, 0.5, 1e-6
    rng = np.random.default_rng(side)
    x = (rng.uniform(0, n, (3, side ** 3)).astype(np.float32)) % np.float32(n)
    v = rng.normal(0, 1e-3, (3, side ** 3)).astype(np.float32)
    # the second member: an undisturbed lattice whose scale factor runs out two steps after the first part
    q = np.arange(16) * 2 + 0.5
    lattice = np.stack([g.ravel() for g in np.meshgrid(q, q, q, indexing="ij")]).astype(np.float32)
    got, want = _member(n, side, x, v), _member(n, side, x, v)
    short = _member(n, 16, lattice, np.zeros_like(lattice))
    ens = PMEnsemble([got, short])
    with pytest.raises(RuntimeError, match="must stay positive"):
        ens.run([a0, (CHUNK + 2.5) * da], [da, -da], CHUNK + 10)
    ref = PMEnsemble([want])
    ref.run([a0], [da], CHUNK)
    for a, b in zip(got.get_state(np.float64), want.get_state(np.float64)):
        assert np.array_equal(a, b)
    ens.close()
    ref.close()
    for s in (got, want, short):
        s.close()
