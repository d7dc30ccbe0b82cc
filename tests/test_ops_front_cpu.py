"""The Python front end of the operators (paella_amd/ops.py): what it hands to the library, without a device."""
import ctypes

import numpy as np
import pytest
import torch

from paella_amd import ops


@pytest.mark.parametrize("kind", [int, ctypes.c_void_p])
def test_a_direct_queue_waits_for_torchs_stream_however_it_is_named(monkeypatch, kind):
    waited = []
    monkeypatch.setattr(ops, "_direct_queues", {0x1000})
    monkeypatch.setattr(ops.torch.cuda, "current_stream", lambda: type("S", (), {"synchronize": lambda self: waited.append(1)})())
    assert ops._stream(kind(0x1000)) == 0x1000 and waited == [1]
    assert ops._stream(kind(0x2000)) == 0x2000 and waited == [1]  # an ordinary stream orders by itself
    assert ops._stream(ctypes.c_void_p(None)) is None and waited == [1]


def test_a_plan_that_is_replaced_is_the_one_that_is_launched(monkeypatch):
    w = np.ones((8, 16, 3, 3), np.float32)
    conv, other = (ops.Conv2d(w, pad=1, in_hw=hw, device="cpu") for hw in ((9, 9), (5, 7)))
    launched = []
    conv._launch = lambda plan, *rest: launched.append((plan._obj.P, plan._obj.Q)) or 0
    monkeypatch.setattr(ops, "_ptr", lambda t: t if t is None else t.data_ptr())
    monkeypatch.setattr(ops, "_stream", lambda stream: stream)
    assert conv(torch.zeros(1, 16, 9, 9)).shape == (1, 8, 9, 9)
    conv.plan = other.plan
    assert conv(torch.zeros(1, 16, 5, 7)).shape == (1, 8, 5, 7)
    assert launched == [(9, 9), (5, 7)]
    with pytest.raises(AssertionError):
        conv(torch.zeros(1, 16, 9, 9))
