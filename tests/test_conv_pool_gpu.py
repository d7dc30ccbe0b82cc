"""A conv and the pool behind it in one launch (csrc/hip/conv_pool.h) at the edges of windows, tiles and reductions: the bits of the two operators."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# C, K, H, W, (R, S), stride, pad, dilation, window, waves of the plan (log2; None: the plan's own)
CASES = [
    (1, 8, 28, 28, (5, 5), 1, 2, 1, (2, 2), None),    # reduction through the offset table, its last chunk a single value
    (8, 16, 14, 14, (5, 5), 1, 2, 1, (3, 3), None),   # pixels behind the last window; waves without a chunk
    (3, 17, 9, 11, (3, 3), 2, 1, 1, (2, 2), None),    # a channel more than a tile, an odd row and column, a stride
    (8, 1, 2, 2, (1, 1), 1, 0, 1, (2, 2), None),      # one window
    (16, 33, 8, 12, (1, 1), 1, 0, 1, (4, 4), None),   # a window that fills the tile
    (24, 20, 7, 13, (3, 3), 1, 1, 1, (1, 2), 3),      # eight windows to a tile
    (8, 16, 11, 9, (1, 7), 1, (0, 3), 1, (3, 1), 3),  # five, one column idle
    (16, 16, 9, 9, (3, 3), 1, 2, 2, (3, 4), 3),       # a window of twelve, a dilated filter
    (2, 30, 10, 10, (3, 3), 1, 1, 1, (2, 4), 1),      # two waves, which finish two registers each
    (8, 256, 16, 16, (1, 1), 1, 0, 1, (2, 2), 2),     # 256 tiles
]


def make(case, rng, ops, act, bias=True):
    c, k, h, w, (r, s), stride, pad, dil, window, kw = case
    wt = rng.standard_normal((k, c, r, s)).astype(np.float32)
    slope = rng.standard_normal(k).astype(np.float32) if act == ops.ACT_PRELU else None
    hint = 0 if kw is None else 1 << 20 | 0x110 | kw
    return ops.Conv2d(wt, rng.standard_normal(k).astype(np.float32) if bias else None, stride=stride, pad=pad, dil=dil, act=act, slope=slope, in_hw=(h, w), tile_hint=hint)


def pooled(ops, conv, x, window, stream=None):
    from paella_amd import _abi
    plan = conv.plan
    d = _abi.PoolDesc(plan.d.K, plan.P, plan.Q, *window, *window, 0, 0, 0, 0, 1)
    assert _abi.ops().paella_conv2d_plan_takes_pool(ctypes.byref(plan), ctypes.byref(d)) == 1
    y = torch.full((1, plan.d.K, plan.P // window[0], plan.Q // window[1]), 7.25, device=x.device)
    ptr = lambda t: None if t is None else t.data_ptr()
    _abi.check(_abi.ops().paella_conv2d_launch_pooled(ctypes.byref(plan), ctypes.byref(d), ptr(x), ptr(conv.blob), ptr(conv.bias), ptr(conv.slope), ptr(y),
                                                      stream or torch.cuda.current_stream().cuda_stream), "paella_conv2d_launch_pooled")
    return y


@pytest.mark.parametrize("case", CASES)
def test_one_launch_gives_the_bits_of_two(cuda, case):
    from paella_amd import ops
    rng = np.random.default_rng(sum(case[:4]))
    for act in (ops.ACT_RELU, ops.ACT_PRELU):
        conv = make(case, rng, ops, act, bias=act != ops.ACT_RELU)
        x = torch.tensor(rng.standard_normal((1, case[0], case[2], case[3])).astype(np.float32), device=cuda)
        want = ops.pool2d(conv(x), case[8], case[8])
        for _ in range(2):
            assert torch.equal(pooled(ops, conv, x, case[8]), want)


def test_values_that_are_no_numbers_take_the_way_of_the_two_operators(cuda):
    from paella_amd import ops
    rng = np.random.default_rng(5)
    conv = make(CASES[1], rng, ops, 0)
    x = rng.standard_normal((1, 8, 14, 14)).astype(np.float32)
    x[0, 1, :4, :4], x[0, 2, 8, 8], x[0, 3, 12, 2] = np.nan, np.inf, -np.inf
    x = torch.tensor(x, device=cuda)
    got, want = pooled(ops, conv, x, (3, 3)), ops.pool2d(conv(x), 3, 3)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32)) and not torch.isfinite(want).all()


def small_file(path):
    """A conv of 8 channels on 28 x 28 and its pool as a file of their own."""
    import _onnx_writer as ow
    b = ow.Builder(np.random.default_rng(3))
    y = b.op("Relu", [b.op("Conv", ["x", b.const(b.randn(8, 1, 5, 5, scale=0.2)), b.const(b.randn(8))], kernel_shape=[5, 5], pads=[2, 2, 2, 2])])
    y = b.op("MaxPool", [y], kernel_shape=[2, 2], strides=[2, 2])
    b.save(str(path), [("x", [1, 1, 28, 28])], [(y, [1, 8, 14, 14])])
    return "onnx:" + str(path)


def test_input_and_output_in_the_same_memory(cuda, tmp_path):
    """Bound to the same memory the two stay two launches: the pool writes over what the conv has read."""
    from paella_amd import models
    ex = models.Exec(small_file(tmp_path / "inplace.onnx"))
    x = torch.tensor(np.random.default_rng(6).standard_normal(784).astype(np.float32), device=cuda)
    apart, same = torch.zeros(1568, device=cuda), torch.zeros(1568, device=cuda)
    ex.bind_io(x.data_ptr(), apart.data_ptr())
    ex.forward()
    ex.bind_io(same.data_ptr(), same.data_ptr())
    for _ in range(3):
        same[:784] = x
        torch.cuda.synchronize()
        ex.forward()
        torch.cuda.synchronize()
        assert torch.equal(same, apart)
    ex.close()


def test_pairs_in_replayed_passes(cuda, tmp_path):
    """Two pairs in a pass that is long enough for a graph: recorded and replayed on several streams, the bits of the stages one by one."""
    import _onnx_writer as ow
    from paella_amd import models
    from test_exec_io_gpu import plain
    b = ow.Builder(np.random.default_rng(9))

    def conv(x, k, c, r):
        return b.op("Relu", [b.op("Conv", [x, b.const(b.randn(k, c, r, r, scale=1.0 / np.sqrt(c) / r)), b.const(b.randn(k))], kernel_shape=[r, r], pads=[r // 2] * 4)])
    y = b.op("MaxPool", [conv("x", 8, 1, 5)], kernel_shape=[2, 2], strides=[2, 2])
    y = b.op("MaxPool", [conv(y, 16, 8, 5)], kernel_shape=[3, 3], strides=[3, 3])
    for _ in range(14):
        y = conv(y, 16, 16, 1)
    b.save(str(tmp_path / "chain.onnx"), [("x", [1, 1, 28, 28])], [(y, [1, 16, 4, 4])])
    name = "onnx:" + str(tmp_path / "chain.onnx")
    assert len(models.launch_plan(name)) == 18
    rng = np.random.default_rng(10)
    xs = [rng.standard_normal(784).astype(np.float32) for _ in range(2)]
    want = [plain(name, x) for x in xs]
    assert not np.array_equal(*want)
    execs, streams = [models.Exec(name) for _ in range(4)], [torch.cuda.Stream() for _ in range(2)]
    other = torch.zeros(1 << 16, device=cuda)
    for turn in range(8):
        for i, ex in enumerate(execs):
            ex.set_input(xs[(i + turn) % 2])
            ex.forward(streams[i % 2].cuda_stream)
        other += 1
        for s in streams:
            s.synchronize()
        for i, ex in enumerate(execs):
            np.testing.assert_array_equal(ex.get_output(), want[(i + turn) % 2])
    for ex in execs:
        ex.close()


@pytest.mark.parametrize("limit", ["6400", "8192", "65536"])
def test_served_with_pairs_within_the_limit_of_small_kernels_and_beyond(cuda, monkeypatch, limit):
    """The small CNN under load with none, one and both of its pairs as one launch: every answer as that of the idle server, and that the oracle's."""
    from paella_amd import models, serve
    from test_verify_gpu import expectations_match_the_oracle, run_verified, server_name
    monkeypatch.setenv("LLIS_MODEL_SEED", "1")
    monkeypatch.setenv("PAELLA_GROUP_THREADS", limit)
    types = [("mnist", "tvm_mnist", 1.0, 48)]
    with serve.Server(server_name("pairs"), "full3", num_streams=32, extra_kernels=32) as srv:
        r, out_bytes = run_verified(serve, models, srv, types, 0.0, 3000, seed=5)
    assert r["mismatches"] == 0
    expectations_match_the_oracle(models, types, r, out_bytes, 5)
