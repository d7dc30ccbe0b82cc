"""Inputs written to device memory by the host (paella_exec_store_input), by the call or by the library's copy thread: the bits of a
pass on the same input copied by the runtime, whatever the request's last input was and whether the thread was awake."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["mnist", "ultraface320", "squeezenet1_1"])
def test_stored_inputs_reach_the_kernels(cuda, name):
    from paella_amd import _abi, models, ops
    hip, rng = _abi.hip(), np.random.default_rng(5)
    ex, plain = models.Exec(name), models.Exec(name)
    n = models.io_bytes(name)[0] // 4
    xs = [rng.standard_normal(n + 3).astype(np.float32)[i:i + n] for i in (0, 1, 3)]  # 64-byte lines and not
    want = []
    for x in xs:
        _abi.check(hip.llis_hip_memcpy(plain.lib.paella_exec_input(plain.handle), np.ascontiguousarray(x).ctypes.data, x.nbytes, 1))
        plain.forward()
        want.append(plain.get_output())
    told = []
    done = ctypes.CFUNCTYPE(None, ctypes.c_void_p)(told.append)
    call = ctypes.cast(done, ctypes.c_void_p)
    with ops.DirectQueue(ordered=True) as q:
        for turn in range(24):
            x = xs[turn * 5 % 3]
            if turn % 4 == 3:
                time.sleep(0.002)  # the copy thread sleeps: the call writes
            by_call = turn % 3 == 0
            _abi.check(ex.lib.paella_exec_store_input(ex.handle, x.ctypes.data, None if by_call else call, None if by_call else turn + 1))
            limit = time.monotonic() + 5
            while not by_call and (not told or told[-1] != turn + 1):
                assert time.monotonic() < limit
            ex.forward(q.handle)
            q.wait()
            np.testing.assert_array_equal(ex.get_output(), want[turn * 5 % 3])
    ex.close()
    plain.close()


def test_memory_the_host_does_not_address_is_refused(cuda):
    from paella_amd import _abi, models
    handle, model = ctypes.c_void_p(), models.Exec("mnist")
    lib = model.lib
    _abi.check(lib.paella_exec_create(model.model, ctypes.byref(handle)))
    x = np.zeros(784, np.float32)
    assert lib.paella_exec_store_input(handle, x.ctypes.data, None, None) == -2
    assert lib.paella_exec_store_input(handle, None, None, None) == -1
    _abi.check(lib.paella_exec_destroy(handle))
    model.close()
