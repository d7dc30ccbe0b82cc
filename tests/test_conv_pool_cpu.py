"""Which convs go out with the pool behind them (host arithmetic; the results: test_conv_pool_gpu.py)."""
import ctypes

import pytest


def conv_plan(c, k, h, w, r, hint=0):
    from paella_amd import _abi
    desc = _abi.ConvDesc(c, h, w, k, r, r, 1, 1, r // 2, r // 2, 1, 1, 1, 1, 0.0, 0.0)
    plan = _abi.ConvPlan()
    assert _abi.ops().paella_conv2d_plan(ctypes.byref(desc), 0, hint, ctypes.byref(plan)) == 0
    return plan


def takes(c, k, h, w, r, pool, pool_stride=None, pool_pad=0, ceil=0, avg=0, hint=0, channels=None):
    from paella_amd import _abi
    lib = _abi.ops()
    plan = conv_plan(c, k, h, w, r, hint)
    s = pool_stride or pool
    d = _abi.PoolDesc(channels or k, h, w, pool, pool, s, s, pool_pad, pool_pad, ceil, avg, 1)
    return lib.paella_conv2d_plan_takes_pool(ctypes.byref(plan), ctypes.byref(d))


@pytest.mark.parametrize("case, want", [
    (dict(c=1, k=8, h=28, w=28, r=5, pool=2), 1), (dict(c=8, k=16, h=14, w=14, r=5, pool=3), 1),
    (dict(c=8, k=16, h=14, w=14, r=5, pool=3, pool_stride=2), 0),        # windows that share pixels
    (dict(c=8, k=16, h=14, w=14, r=5, pool=2, pool_pad=1), 0), (dict(c=8, k=16, h=14, w=14, r=5, pool=2, ceil=1), 0),
    (dict(c=8, k=16, h=14, w=14, r=5, pool=2, avg=1), 0), (dict(c=8, k=16, h=14, w=14, r=5, pool=5), 0),
    (dict(c=8, k=16, h=2, w=14, r=5, pool=3), 0),                        # a window larger than the image
    (dict(c=8, k=16, h=14, w=14, r=5, pool=2, channels=8), 0),           # another tensor's pool
    (dict(c=56, k=16, h=14, w=14, r=3, pool=2, hint=1 << 20 | 0x113), 1), (dict(c=64, k=16, h=14, w=14, r=3, pool=2, hint=1 << 20 | 0x113), 0),  # eight and nine chunks per wave
    (dict(c=64, k=16, h=14, w=14, r=3, pool=2, hint=1 << 20 | 0x1113), 0),  # a split reduction
    (dict(c=8, k=256, h=16, w=16, r=1, pool=2), 1), (dict(c=8, k=272, h=16, w=16, r=1, pool=2), 0),  # 256 tiles and 272
    (dict(c=8, k=16, h=14, w=14, r=5, pool=2, hint=0x113), 0),           # a plan whose form is given
])
def test_which_convs_take_their_pool(case, want):
    assert takes(**case) == want


@pytest.mark.parametrize("window", [(0, 0), (0, 2), (2, 0), (-1, -2), (-2, -2), (2, -2)])
def test_a_pool_that_is_none_is_refused(window):
    """As the pool's own entry points refuse it."""
    from paella_amd import _abi
    lib = _abi.ops()
    plan = conv_plan(8, 16, 14, 14, 5)
    memory = ctypes.c_void_p(4096)  # never looked at
    d = _abi.PoolDesc(16, 14, 14, *window, *window, 0, 0, 0, 0, 1)
    assert lib.paella_conv2d_plan_takes_pool(ctypes.byref(plan), ctypes.byref(d)) == 0
    assert lib.paella_conv2d_launch_pooled(ctypes.byref(plan), ctypes.byref(d), memory, memory, None, None, ctypes.c_void_p(1 << 20), None) == -2
    assert lib.paella_pool2d_dims(ctypes.byref(d), ctypes.byref(_abi.LaunchDims())) != 0


@pytest.mark.parametrize("x, y", [(1 << 20, 1 << 20), (1 << 20, (1 << 20) + 8 * 14 * 14 * 4 - 4), ((1 << 20) + 16 * 4 * 4 * 4 - 4, 1 << 20)])
def test_an_output_that_lies_in_the_input_is_refused(x, y):
    """Workgroups that have their windows write while others still read: two launches can do that, one cannot."""
    from paella_amd import _abi
    plan = conv_plan(8, 16, 14, 14, 5)
    d = _abi.PoolDesc(16, 14, 14, 3, 3, 3, 3, 0, 0, 0, 0, 1)
    ptr = ctypes.c_void_p
    assert _abi.ops().paella_conv2d_plan_takes_pool(ctypes.byref(plan), ctypes.byref(d)) == 1
    assert _abi.ops().paella_conv2d_launch_pooled(ctypes.byref(plan), ctypes.byref(d), ptr(x), ptr(4096), None, None, ptr(y), None) == -2
