"""A request run by itself: in the grid's own tile shape unless the caller names one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _request(n, n_parts):
    from pmgpu.serve import SimRequest
    return SimRequest(id=n, seed=3, box=2.0 * n, n_cells=n, n_parts=n_parts, steps=12)


@pytest.mark.parametrize("n", [16, 32, 64, 128])
@pytest.mark.parametrize("tiles", [None, (8, 8, 8)])
def test_shape_of_a_lone_run(n, tiles, monkeypatch):
    from pmgpu import serve
    from pmgpu.sim import PMSim
    seen = []

    class Watched(PMSim):
        def run(self, *args):
            seen.append(self.tiles())
            return super().run(*args)

    monkeypatch.setattr(serve, "PMSim", Watched)
    q = _request(n, n // 2)
    r = serve.run_alone(q, keep_state=True, tiles=tiles)
    plain = PMSim(n, q.n_parts, 32)
    assert seen == [tiles or plain.tiles()]
    plain.close()
    assert r.steps == q.loop_steps and r.error is None
    assert np.isfinite(r.positions).all() and np.isfinite(r.velocities).all() and np.isfinite(r.pk[1:2]).all()
