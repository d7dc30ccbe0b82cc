"""When the executor records a pass (paella_exec_forward), which convs go out with the pool behind them, on the scripted device, and the host's
copies: tests/fake_device/exec_check.cpp."""
import os
import subprocess

import numpy as np
import pytest

import _onnx_writer as ow
from _fake import FAKE_LIB, ensure_built
from paella_amd import models


def counts(how):
    ensure_built()
    out = subprocess.run([os.path.join(FAKE_LIB, "exec_check"), how], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    return [tuple(int(v) for v in line.split()) for line in out.stdout.splitlines()]


def test_a_pass_that_cannot_be_recorded_is_tried_once_per_buffers():
    """Ten passes of each of two requests, then ten more on other input memory: (recordings tried, plain passes, replayed passes)."""
    assert counts("refuse") == [(2, 20, 0), (4, 40, 0)]


def test_the_fourth_pass_in_company_is_recorded():
    """(A pass that this machine holds up for 150 us is not in company and goes out plain.)"""
    for turn, (recorded, plain, replayed) in enumerate(counts("allow"), 1):
        assert recorded == 2 * turn and plain >= 6 * turn and replayed > 0 and plain + replayed == 20 * turn


def test_host_copies_touch_their_bytes_and_no_others():
    assert counts("copies") == [(19,)]


def launches(model, ranges, takes="takes", **env):
    """What paella_exec_launch_stages returns and issues for each (first, last, with a notifier)."""
    ensure_built()
    args = [str(int(v)) for r in ranges for v in r]
    out = subprocess.run([os.path.join(FAKE_LIB, "exec_check"), "launches", model, takes] + args, capture_output=True, text=True, timeout=60, env=dict(os.environ, **env))
    assert out.returncode == 0, out.stderr
    return out.stdout.splitlines()


CNN = [(0, 4, 0), (0, 4, 1), (0, 0, 0), (0, 1, 0), (0, 1, 1), (0, 2, 1), (1, 3, 0), (1, 3, 1), (2, 3, 0), (1, 1, 1), (3, 4, 1)]


def test_stages_in_order_share_a_launch_within_a_range_whose_pool_reports_to_nobody():
    want = ["0 pooled pooled 4", "0 pooled pooled 4*7", "0 0", "0 pooled", "0 0 1*7", "0 pooled 2*7", "0 1 pooled", "0 1 2 3*7", "0 pooled", "0 1*7", "0 3 4*7"]
    assert launches("mnist", CNN) == want


def test_a_pair_that_is_refused_is_two_launches():
    want = ["0 " + " ".join(str(k) for k in range(first, last + 1)) + ("*7" if notifier else "") for first, last, notifier in CNN]
    assert launches("mnist", CNN, "refuses") == want
    assert launches("mnist", CNN, PAELLA_CONV_PAIRS="0") == want


@pytest.mark.parametrize("first, last", [(-1, 1), (1, 0), (0, 5), (5, 5), (-2, -1)])
def test_a_range_that_is_none_is_refused(first, last):
    assert launches("mnist", [(first, last, 0)]) == ["-1"]


def conv(b, x, k, c, r=3, act="Relu"):
    y = b.op("Conv", [x, b.const(b.randn(k, c, r, r, scale=0.1)), b.const(b.randn(k))], kernel_shape=[r, r], pads=[r // 2] * 4)
    return b.op(act, [y]) if act else y


def pool(b, x, r=2, stride=None, op="MaxPool", **attrs):
    return b.op(op, [x], kernel_shape=[r, r], strides=[stride or r] * 2, **attrs)


def head(b, x):
    return b.op("Flatten", [b.op("GlobalAveragePool", [x])])


def graph_plain(b):
    return head(b, pool(b, conv(b, "x", 16, 8))), [1, 16]


def graph_second_reader(b):
    c = conv(b, "x", 16, 8)
    return b.op("Add", [head(b, pool(b, c)), head(b, c)]), [1, 16]


def graph_output_is_the_convs(b):
    c = conv(b, "x", 16, 8)
    pool(b, c)
    return c, [1, 16, 12, 12]


def graph_output_is_read(b):
    """The conv's input is the graph's output, which can be bound to memory of the caller."""
    a = conv(b, "x", 16, 8)
    pool(b, conv(b, a, 16, 16))
    return a, [1, 16, 12, 12]


def graph_slice_of_a_concatenation(b):
    """The conv's output is a part of what the concatenation's reader reads."""
    c = conv(b, "x", 16, 8)
    p = pool(b, c)
    return b.op("Concat", [head(b, p), head(b, b.op("Concat", [c, "x"], axis=1))], axis=1), [1, 40]


def graph_pool_of_a_concatenation(b):
    """The pool reads more than the conv in front of it wrote."""
    a = conv(b, "x", 16, 8)
    both = b.op("Concat", [conv(b, a, 16, 16), a], axis=1)
    return head(b, pool(b, both)), [1, 32]


def graph_pool_into_a_concatenation(b):
    """What the pool writes lies beside another result."""
    c = pool(b, conv(b, "x", 16, 8))
    return head(b, b.op("Concat", [b.op("LRN", [c], size=3), c], axis=1)), [1, 32]


def graph_residual(b):
    a = conv(b, "x", 16, 8)
    c = b.op("Relu", [b.op("Add", [conv(b, a, 16, 16, act=None), a])])
    return head(b, pool(b, c)), [1, 16]


def graph_transformed_input(b):
    """A batch normalisation that the conv applies to its own input."""
    a = conv(b, "x", 16, 8)
    n = b.op("Relu", [b.op("BatchNormalization", [pool(b, a, op="AveragePool")] + [b.const(np.abs(b.randn(16)) + 0.5) for _ in range(4)])])
    return head(b, pool(b, conv(b, n, 16, 16))), [1, 16]


def graph_two_convs_in_a_launch(b):
    c = conv(b, "x", 16, 8, 5)
    other = conv(b, "x", 16, 8)
    return b.op("Add", [head(b, pool(b, c)), head(b, other)]), [1, 16]


def graph_a_pool_in_the_convs_launch(b):
    c = conv(b, "x", 8, 8)
    other = pool(b, "x", 3, 1, op="AveragePool", pads=[1] * 4)
    return b.op("Add", [head(b, pool(b, c)), head(b, other)]), [1, 8]


def graph_average(b):
    return head(b, pool(b, conv(b, "x", 16, 8), op="AveragePool")), [1, 16]


@pytest.mark.parametrize("graph, pairs", [
    (graph_plain, 1), (graph_pool_into_a_concatenation, 1), (graph_second_reader, 0), (graph_output_is_the_convs, 0), (graph_slice_of_a_concatenation, 0),
    (graph_pool_of_a_concatenation, 0), (graph_residual, 0), (graph_transformed_input, 0), (graph_average, 0), (graph_output_is_read, 0),
    (graph_two_convs_in_a_launch, 0), (graph_a_pool_in_the_convs_launch, 0),
], ids=lambda v: v.__name__[6:] if callable(v) else str(v))
def test_which_convs_of_a_graph_leave_their_output_unwritten(tmp_path, graph, pairs):
    """Those whose output the next stage, a pool, reads and nothing else."""
    b = ow.Builder(np.random.default_rng(7))
    y, shape = graph(b)
    path = str(tmp_path / "g.onnx")
    b.save(path, [("x", [1, 8, 12, 12])], [(y, shape)])
    model = "onnx:" + path
    count = len(models.launch_plan(model))
    issued = launches(model, [(0, count - 1, 0)])[0].split()
    assert issued[0] == "0" and issued[1:].count("pooled") == pairs and len(issued) - 1 == count - pairs


@pytest.mark.parametrize("channels, window, want", [(24, 2, "pooled"), (32, 2, "0 1"), (24, 3, "pooled"), (56, 3, "0 1"), (32, 4, "pooled"), (56, 4, "pooled"), (64, 4, "0 1")])
def test_convs_of_more_than_four_chunks_per_wave_keep_a_launch_of_their_own(tmp_path, channels, window, want):
    """Unless the windows fill the tiles.  (Four, five, eight and nine chunks in each of eight waves.)"""
    b = ow.Builder(np.random.default_rng(8))
    y = pool(b, conv(b, "x", 32, channels), window)
    path = str(tmp_path / "g.onnx")
    b.save(path, [("x", [1, channels, 30, 30])], [(y, [1, 32, 30 // window, 30 // window])])
    assert launches("onnx:" + path, [(0, 1, 0)]) == ["0 " + want]
