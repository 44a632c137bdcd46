"""pm_malloc / pm_free: freed blocks are handed out again, freed memory is reported as free, and a
block is never handed out twice."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _malloc(nbytes):
    from pmgpu import _lib
    _lib.init()
    p = C.c_void_p()
    _lib.call("pm_malloc", C.byref(p), nbytes)
    return p


def _free(p):
    from pmgpu import _lib
    _lib.call("pm_free", p)


def _free_bytes():
    from pmgpu.serve import device_memory
    return device_memory()[0]


@pytest.mark.parametrize("nbytes", [0, 1, 64 << 10, (64 << 10) + 1, 3 * MIB + 5, 64 * MIB])
def test_a_freed_block_serves_the_next_request_of_its_size(nbytes):
    p, q = _malloc(nbytes), _malloc(nbytes)
    assert p.value != q.value
    a = p.value
    _free(p)
    r = _malloc(nbytes)
    assert r.value == a and r.value != q.value
    _free(q)
    _free(r)


def test_freed_memory_counts_as_free_and_a_second_free_is_refused():
    before = _free_bytes()
    p = _malloc(512 * MIB)
    a = p.value
    assert _free_bytes() <= before - 500 * MIB
    _free(p)
    with pytest.raises(RuntimeError):
        _free(C.c_void_p(a))
    assert _free_bytes() >= before - 8 * MIB   # the report gives kept blocks back first


def test_threads_get_blocks_of_their_own():
    from pmgpu.device import DeviceArray
    bad = []

    def work(i):
        for k in range(20):
            d = DeviceArray.from_numpy(np.full(1 << 18, 100 * i + k, np.int32))
            if not (d.numpy() == 100 * i + k).all():
                bad.append((i, k))
            del d

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
