"""Memory that a density() or integrate() call uses for its tile bins counts as free once the call is
over: the next sim, or a serving budget, gets it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _free_bytes():
    from pmgpu.serve import device_memory
    return device_memory()[0]


@pytest.mark.parametrize("what", ["density", "integrate"])
def test_bins_of_a_call_are_reported_as_free(what):
    from pmgpu import ops
    from pmgpu.device import DeviceArray
    n, n_p = 128, 1 << 22                                # bins of about 135 MB, or 17 of own entries alone
    x = DeviceArray.from_numpy((np.random.default_rng(1).uniform(0, n, (3, n_p)) % n).astype(np.float32) % np.float32(n))
    v = DeviceArray.zeros((3, n_p), np.float32)
    phi = DeviceArray.zeros((n, n, n), np.float32)
    before = _free_bytes()
    for _ in range(2):
        if what == "density":
            del_me = ops.density(x, 1.0, n)
            del del_me
        else:
            ops.integrate(x, v, 0.5, 1.0, 0.01, phi, n)
        assert _free_bytes() >= before - 8 * MIB
