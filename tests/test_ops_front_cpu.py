"""The Python front end of the operators (paella_amd/ops.py): what it hands to the library, without a device."""
import ctypes

import pytest

from paella_amd import ops


@pytest.mark.parametrize("kind", [int, ctypes.c_void_p])
def test_a_direct_queue_waits_for_torchs_stream_however_it_is_named(monkeypatch, kind):
    waited = []
    monkeypatch.setattr(ops, "_direct_queues", {0x1000})
    monkeypatch.setattr(ops.torch.cuda, "current_stream", lambda: type("S", (), {"synchronize": lambda self: waited.append(1)})())
    assert ops._stream(kind(0x1000)) == 0x1000 and waited == [1]
    assert ops._stream(kind(0x2000)) == 0x2000 and waited == [1]  # an ordinary stream orders by itself
    assert ops._stream(ctypes.c_void_p(None)) is None and waited == [1]
