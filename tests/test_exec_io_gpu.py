"""Host input and output of a request (paella_exec_host_io) and replayed passes (csrc/hip/forward_graph.h): the bits of one plain pass,
however often, on whatever streams and between whatever other work the passes run."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def plain(name, x):
    """One pass stage by stage, its input and output moved by the runtime's copies through the addresses the request names."""
    from paella_amd import _abi, models
    ex = models.Exec(name)
    hip = _abi.hip()
    _abi.check(hip.llis_hip_memcpy(ex.lib.paella_exec_input(ex.handle), x.ctypes.data, x.nbytes, 1))
    for i in range(ex.num_stages):
        ex.launch_stage(i)
    out = np.empty(ex.out_bytes // 4, np.float32)
    _abi.check(hip.llis_hip_memcpy(out.ctypes.data, ex.lib.paella_exec_output(ex.handle), out.nbytes, 2))
    ex.close()
    return out


@pytest.mark.parametrize("name", ["mnist", "squeezenet1_1", "ultraface320"])
def test_replayed_passes_on_several_streams_give_the_bits_of_one_plain_pass(cuda, name):
    from paella_amd import models
    rng = np.random.default_rng(7)
    n = 6
    xs = [rng.standard_normal(models.io_bytes(name)[0] // 4).astype(np.float32) for _ in range(2)]
    want = [plain(name, x) for x in xs]
    execs, streams = [models.Exec(name) for _ in range(n)], [torch.cuda.Stream() for _ in range(3)]
    other = torch.zeros(1 << 16, device=cuda)
    for turn in range(8):
        for i, ex in enumerate(execs):
            ex.set_input(xs[(i + turn) % 2])
            ex.forward(streams[i % 3].cuda_stream)
        other += 1  # eager work between the passes, also on one of their streams
        with torch.cuda.stream(streams[0]):
            other.mul_(1.0)
        for s in streams:
            s.synchronize()
        for i, ex in enumerate(execs):
            np.testing.assert_array_equal(ex.get_output(), want[(i + turn) % 2])
    for _ in range(20):  # back to back on one stream: each pass behind the one before
        execs[0].forward(streams[1].cuda_stream)
    streams[1].synchronize()
    np.testing.assert_array_equal(execs[0].get_output(), want[7 % 2])
    for ex in execs:
        ex.close()


def test_buffers_that_move_and_a_stream_that_is_gone(cuda):
    """Bound memory takes over from the request's own and gives it back; a graph recorded before is not used for the other buffers.  The
    stream of the last pass may be destroyed before the next pass."""
    from paella_amd import _abi, models
    name = "squeezenet1_1"
    hip, rng = _abi.hip(), np.random.default_rng(8)
    x, y = (rng.standard_normal(models.io_bytes(name)[0] // 4).astype(np.float32) for _ in range(2))
    want_x, want_y = plain(name, x), plain(name, y)
    busy, ex = models.Exec(name), models.Exec(name)
    host_in, host_out = ctypes.c_void_p(), ctypes.c_void_p()
    _abi.check(hip.llis_hip_host_alloc_pinned(ctypes.byref(host_in), ex.in_bytes))
    _abi.check(hip.llis_hip_host_alloc_pinned(ctypes.byref(host_out), ex.out_bytes))
    busy.set_input(y)
    ex.set_input(x)
    for bound in (False, True, False):
        ex.bind_io(host_in.value if bound else None, host_out.value if bound else None)
        if bound:
            ctypes.memmove(host_in, y.ctypes.data, y.nbytes)
        for _ in range(6):
            s = ctypes.c_void_p()
            _abi.check(hip.llis_hip_stream_create(ctypes.byref(s)))
            busy.forward(s)
            ex.forward(s)
            _abi.check(hip.llis_hip_stream_synchronize(s))
            _abi.check(hip.llis_hip_stream_destroy(s))
            np.testing.assert_array_equal(ex.get_output(), want_y if bound else want_x)
            np.testing.assert_array_equal(busy.get_output(), want_y)
    ex.close()
    busy.close()
    hip.llis_hip_host_free(host_in)
    hip.llis_hip_host_free(host_out)


def test_inputs_off_the_lines_of_a_streaming_store_and_memory_of_earlier_requests(cuda):
    """Inputs of odd sizes and addresses, outputs of 40 to 35 360 bytes; what an earlier request left behind never shows."""
    from paella_amd import models
    rng = np.random.default_rng(9)
    for turn in range(3):
        for name in ("mnist", "ultraface320", "arcfaceresnet100"):
            ex = models.Exec(name)
            x = rng.standard_normal(ex.in_bytes // 4 + 1).astype(np.float32)[1:]  # four bytes past a line
            ex.set_input(x)
            ex.forward()
            np.testing.assert_array_equal(ex.get_output(), plain(name, np.ascontiguousarray(x)))
            ex.close()


@pytest.mark.parametrize("name", ["mnist", "squeezenet1_1"])
def test_input_and_output_wait_for_passes_on_a_blocking_stream(cuda, name):
    """Where the host moves them itself they wait for what a copy on the null stream waits for: a pass still queued on a stream that
    orders with it, behind 20 ms of other work."""
    from paella_amd import _abi, models
    hip, rng = _abi.hip(), np.random.default_rng(10)
    x, y = (rng.standard_normal(models.io_bytes(name)[0] // 4).astype(np.float32) for _ in range(2))
    want_x, want_y = plain(name, x), plain(name, y)
    busy, ex = models.Exec("arcfaceresnet100"), models.Exec(name)
    s = ctypes.c_void_p()
    _abi.check(hip.hipStreamCreate(ctypes.byref(s)))
    busy.set_input(np.zeros(busy.in_bytes // 4, np.float32))
    for _ in range(3):  # past the inputs that the runtime copies
        ex.set_input(x)
        ex.forward(s)
        np.testing.assert_array_equal(ex.get_output(), want_x)
    for late in (False, True):
        ex.set_input(y)
        for _ in range(20):
            busy.forward(s)
        ex.forward(s)
        if late:
            ex.set_input(x)  # not under the pass that reads y
        np.testing.assert_array_equal(ex.get_output(), want_y)
        ex.forward(s)
        np.testing.assert_array_equal(ex.get_output(), want_x if late else want_y)
    _abi.check(hip.llis_hip_stream_destroy(s))
    ex.close()
    busy.close()
