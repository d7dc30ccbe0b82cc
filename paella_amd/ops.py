"""Functional front-end over the operator C-ABI for tests and benches.

Tensors are torch CUDA tensors (torch is only the allocator and stream provider here); weights are packed
on the host with paella_conv2d_pack and uploaded.  Everything runs on the calling thread's current torch
stream unless a stream handle is given.
"""
import ctypes
import functools

import numpy as np
import torch

from . import _abi
from ._abi import ConvDesc, ConvOperands, ConvPlan, LaunchDims, PoolDesc, check

ACT_NONE, ACT_RELU, ACT_RELU6, ACT_PRELU, ACT_CLIP = range(5)


# A call's time on a small layer is what it costs the calling thread: the launch is 2.7 us of it, an output tensor 1.2, and everything
# here is meant to stay under 1 (torch.cuda.current_stream alone is 2.6; pointers go to the library as plain integers).

def _ptr(t):
    if t is None:
        return None
    assert t.is_cuda and t.dtype == torch.float32 and t.is_contiguous()
    return t.data_ptr()


def _torch_stream():
    return torch.cuda.current_stream().cuda_stream


try:
    from torch._C import _cuda_getCurrentRawStream, _cuda_getDevice

    def _torch_stream():  # noqa: F811  (the same handle without the stream object around it)
        return _cuda_getCurrentRawStream(_cuda_getDevice())
except ImportError:
    pass


_direct_queues = set()


def _stream(stream):
    if stream is None:
        return _torch_stream()
    if isinstance(stream, ctypes.c_void_p):
        stream = stream.value
    if stream in _direct_queues:
        # nothing orders such a queue behind torch's stream, and a call is quick enough to overtake a fill that is still under way there
        torch.cuda.current_stream().synchronize()
    return stream


def _pair(v):
    return (v, v) if isinstance(v, int) else tuple(v)


class Conv2d:
    """One planned conv layer: packed weights resident on the device."""

    def __init__(self, w, bias=None, stride=1, pad=0, dil=1, groups=1, act=ACT_NONE, lo=0.0, hi=0.0,
                 in_hw=None, has_residual=False, slope=None, tile_hint=0, device="cuda:0"):
        lib = _abi.ops()
        w = np.ascontiguousarray(w, dtype=np.float32)
        k, cg, r, s = w.shape
        sh, sw = _pair(stride)
        ph, pw = _pair(pad)
        dh, dw = _pair(dil)
        h, wd = in_hw
        self.desc = ConvDesc(cg * groups, h, wd, k, r, s, sh, sw, ph, pw, dh, dw, groups, act, lo, hi)
        plan = ConvPlan()
        check(lib.paella_conv2d_plan(ctypes.byref(self.desc), int(has_residual), tile_hint, ctypes.byref(plan)), "paella_conv2d_plan")
        self.plan = plan
        blob = np.zeros(self.plan.blob_bytes, dtype=np.uint8)
        check(lib.paella_conv2d_pack(ctypes.byref(self.plan), w.ctypes.data, blob.ctypes.data), "paella_conv2d_pack")
        self.blob = torch.from_numpy(blob).to(device)
        self.bias = None if bias is None else torch.tensor(np.asarray(bias, np.float32), device=device)
        self.slope = None if slope is None else torch.tensor(np.asarray(slope, np.float32), device=device)
        self.workspace = torch.zeros(max(self.plan.workspace_bytes, 4) // 4, dtype=torch.int32, device=device) if self.plan.workspace_bytes else None
        self.lib = lib
        self._launch, self._launch_transformed = lib.paella_conv2d_launch, lib.paella_conv2d_launch_transformed

    @property
    def plan(self):
        return self._plan

    @plan.setter
    def plan(self, plan):
        # what every call passes on, looked up once per plan (its extents are not changed in place)
        self._plan, self._plan_ref = plan, ctypes.byref(plan)
        self._in_shape, self._out_shape = (1, plan.d.C, plan.d.H, plan.d.W), (1, plan.d.K, plan.P, plan.Q)

    def takes_input_transform(self):
        return bool(self.lib.paella_conv2d_plan_takes_input_transform(ctypes.byref(self.plan)))

    def __call__(self, x, residual=None, out=None, stream=None, job_id=0, notifier=None, in_scale=None, in_shift=None, in_act=ACT_NONE):
        """in_scale / in_shift (per input channel, device tensors): the conv reads in_act(x * in_scale + in_shift), padded
        with zeros after that transform."""
        assert x.shape == self._in_shape, (tuple(x.shape), self._in_shape)
        y = out if out is not None else x.new_empty(self._out_shape, dtype=torch.float32)
        workspace = self.workspace
        if workspace is not None:
            workspace = workspace.data_ptr()
        if in_scale is not None:
            p = self.plan
            assert in_scale.numel() == p.d.C and in_shift.numel() == p.d.C
            rc = self._launch_transformed(self._plan_ref, _ptr(x), _ptr(in_scale), _ptr(in_shift), in_act, self.blob.data_ptr(), _ptr(self.bias),
                                          _ptr(residual), _ptr(self.slope), _ptr(y), workspace, _stream(stream), job_id, notifier)
            if rc:
                check(rc, "paella_conv2d_launch_transformed")
            return y
        rc = self._launch(self._plan_ref, _ptr(x), self.blob.data_ptr(), _ptr(self.bias), _ptr(residual), _ptr(self.slope), _ptr(y), workspace,
                          _stream(stream), job_id, notifier)
        if rc:
            check(rc, "paella_conv2d_launch")
        return y

    def operands(self, x, residual=None, out=None):
        p = self.plan
        assert x.shape == (1, p.d.C, p.d.H, p.d.W), (tuple(x.shape), p.d.C, p.d.H, p.d.W)
        y = out if out is not None else torch.empty((1, p.d.K, p.P, p.Q), device=x.device, dtype=torch.float32)
        ops = ConvOperands(ctypes.pointer(p), _ptr(x), self.blob.data_ptr(), _ptr(self.bias), _ptr(residual), _ptr(self.slope), _ptr(y),
                           None if self.workspace is None else self.workspace.data_ptr())
        return ops, y


def conv2d_pair(first, x1, second, x2, residual1=None, residual2=None, stream=None, job_id=0, notifier=None):
    """Two independent Conv2d layers as one launch (paella_conv2d_launch_pair); returns both outputs."""
    a, y1 = first.operands(x1, residual1)
    b, y2 = second.operands(x2, residual2)
    check(first.lib.paella_conv2d_launch_pair(ctypes.byref(a), ctypes.byref(b), _stream(stream), job_id, notifier), "paella_conv2d_launch_pair")
    return y1, y2


def conv2d_group(convs, xs, residuals=None, stream=None, job_id=0, notifier=None):
    """Up to four independent Conv2d layers as one launch (paella_conv2d_launch_group); returns their outputs."""
    residuals = residuals or [None] * len(convs)
    members = (ConvOperands * len(convs))()
    outs = []
    for k, (c, x, r) in enumerate(zip(convs, xs, residuals)):
        members[k], y = c.operands(x, r)
        outs.append(y)
    check(convs[0].lib.paella_conv2d_launch_group(members, len(convs), _stream(stream), job_id, notifier), "paella_conv2d_launch_group")
    return outs


def conv2d_group_pool(convs, xs, pool_x, k, stride, pad=0, ceil_mode=False, is_avg=False, count_include_pad=True, residuals=None,
                      stream=None, job_id=0, notifier=None):
    """Up to three independent Conv2d layers and one pooling operator as one launch (paella_conv2d_launch_group_pool);
    returns the convs' outputs and the pool's."""
    residuals = residuals or [None] * len(convs)
    members = (ConvOperands * len(convs))()
    outs = []
    for i, (c, x, r) in enumerate(zip(convs, xs, residuals)):
        members[i], y = c.operands(x, r)
        outs.append(y)
    lib = convs[0].lib
    d, shape = _pool_desc(*pool_x.shape[1:], _pair(k), _pair(stride), _pair(pad), bool(ceil_mode), bool(is_avg), bool(count_include_pad))
    pool_y = torch.empty(shape, device=pool_x.device, dtype=torch.float32)
    check(lib.paella_conv2d_launch_group_pool(members, len(convs), ctypes.byref(d), _ptr(pool_x), _ptr(pool_y), _stream(stream), job_id,
                                              notifier), "paella_conv2d_launch_group_pool")
    return outs, pool_y


def pair_dims(first, second):
    d = LaunchDims()
    rc = first.lib.paella_conv2d_pair_dims(ctypes.byref(first.plan), ctypes.byref(second.plan), ctypes.byref(d))
    return rc, d


@functools.lru_cache(maxsize=256)
def _pool_desc(c, h, w, k, stride, pad, ceil_mode, is_avg, count_include_pad):
    """The descriptor of a pooling operator and the shape of its output."""
    lib = _abi.ops()
    d = PoolDesc(c, h, w, *k, *stride, *pad, int(ceil_mode), int(is_avg), int(count_include_pad))
    return d, (1, c, lib.paella_pool_out(h, k[0], stride[0], pad[0], int(ceil_mode)), lib.paella_pool_out(w, k[1], stride[1], pad[1], int(ceil_mode)))


def dense(x, w, bias=None, act=ACT_NONE, stream=None, job_id=0, notifier=None):
    lib = _abi.ops()
    o, i = w.shape
    y = x.new_empty((1, o), dtype=torch.float32)
    check(lib.paella_dense_launch(_ptr(x), _ptr(w), _ptr(bias), _ptr(y), i, o, act, _stream(stream), job_id, notifier),
          "paella_dense_launch")
    return y


def pool2d(x, k, stride, pad=0, ceil_mode=False, is_avg=False, count_include_pad=True, stream=None, job_id=0,
           notifier=None):
    lib = _abi.ops()
    d, shape = _pool_desc(*x.shape[1:], _pair(k), _pair(stride), _pair(pad), bool(ceil_mode), bool(is_avg), bool(count_include_pad))
    y = x.new_empty(shape, dtype=torch.float32)
    check(lib.paella_pool2d_launch(ctypes.byref(d), _ptr(x), _ptr(y), _stream(stream), job_id, notifier),
          "paella_pool2d_launch")
    return y


def global_avgpool(x, stream=None, job_id=0, notifier=None):
    lib = _abi.ops()
    _, c, h, w = x.shape
    y = torch.empty((1, c, 1, 1), device=x.device, dtype=torch.float32)
    check(lib.paella_global_avgpool_launch(_ptr(x), _ptr(y), c, h * w, _stream(stream), job_id, notifier),
          "paella_global_avgpool_launch")
    return y


def eltwise(a, b=None, scale=None, shift=None, slope=None, act=ACT_NONE, lo=0.0, hi=0.0, stream=None, job_id=0,
            notifier=None):
    lib = _abi.ops()
    c = a.shape[1]
    y = torch.empty_like(a)
    check(lib.paella_eltwise_launch(_ptr(a), _ptr(b), _ptr(scale), _ptr(shift), _ptr(slope), _ptr(y), c,
                                    a.numel() // c, act, lo, hi, _stream(stream), job_id, notifier),
          "paella_eltwise_launch")
    return y


def copy(x, stream=None, job_id=0, notifier=None):
    lib = _abi.ops()
    y = torch.empty_like(x)
    check(lib.paella_copy_launch(_ptr(x), _ptr(y), x.numel(), _stream(stream), job_id, notifier), "paella_copy_launch")
    return y


def softmax(x, stream=None, job_id=0, notifier=None):
    lib = _abi.ops()
    cols = x.shape[-1]
    y = torch.empty_like(x)
    check(lib.paella_softmax_launch(_ptr(x), _ptr(y), x.numel() // cols, cols, _stream(stream), job_id, notifier),
          "paella_softmax_launch")
    return y


def lrn(x, size, alpha, beta, k, stream=None, job_id=0, notifier=None):
    lib = _abi.ops()
    c = x.shape[1]
    y = torch.empty_like(x)
    check(lib.paella_lrn_launch(_ptr(x), _ptr(y), c, x.numel() // c, size, alpha, beta, k, _stream(stream), job_id,
                                notifier), "paella_lrn_launch")
    return y


class DirectQueue:
    """A user-mode hardware queue of the operator library; pass `.handle` as `stream=` to any launch."""

    def __init__(self, ordered=False):
        self.lib = _abi.ops()
        h = ctypes.c_void_p()
        check(self.lib.paella_direct_queue_create(ctypes.byref(h)), "paella_direct_queue_create")
        self.handle = h.value
        _direct_queues.add(self.handle)
        if ordered:
            check(self.lib.paella_direct_queue_set_ordered(h, 1), "paella_direct_queue_set_ordered")

    def wait(self):
        check(self.lib.paella_direct_queue_wait(ctypes.c_void_p(self.handle)), "paella_direct_queue_wait")

    def close(self):
        if self.handle:
            _direct_queues.discard(self.handle)
            check(self.lib.paella_direct_queue_destroy(ctypes.c_void_p(self.handle)), "paella_direct_queue_destroy")
            self.handle = None

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()
