"""Workgroups of two 32 x 32 tiles (conv_tall_tile): the bits of workgroups of one, alone and packed, and each job's notifier sees the
workgroups that its plan counts."""
import ctypes

import numpy as np
import pytest
import torch

from test_conv_small_gpu import reference, rnd
from test_pack_gpu import NO_START, ring  # noqa: F401
from test_ring_gpu import decode

pytestmark = pytest.mark.gpu

# C, K, H, W, (R, S), stride, pad, tile hint (0: the plan's own choice of waves and splits)
EDGES = [
    (64, 33, 1, 1, (1, 1), 1, 0, 0x0113),     # a second tile of one row, one pixel, a chunk per wave
    (72, 64, 5, 7, (1, 1), 1, 0, 0x0113),     # nine chunks over eight waves of two: three of them without any
    (64, 65, 4, 8, (3, 3), 1, 1, 0),          # three tiles: the last rows are a single one
    (64, 96, 11, 3, (3, 3), 1, 1, 0x2113),    # ... with the reduction split four ways; 33 pixels
    (128, 128, 9, 9, (3, 3), 2, 1, 0x1113),   # paired filter columns, two splits
    (128, 160, 8, 8, (3, 3), 2, 0, 0),
    (96, 100, 9, 9, (1, 7), 1, (0, 3), 0),
    (96, 64, 11, 11, (1, 1), 2, 0, 0),        # pointwise with a stride
    (512, 128, 7, 7, (3, 3), 1, 1, 0),        # the plan's own eight splits
    (3, 64, 31, 33, (7, 7), 2, 3, 0),         # the offset table, four waves
    (5, 65, 9, 11, (3, 3), 1, 1, 0x0112),     # ... 45 values: six chunks; a last row of tiles by itself
    (3, 96, 13, 13, (5, 5), 1, 2, 0x1112),    # ... two splits
]


@pytest.mark.parametrize("case", EDGES)
def test_two_tiles_give_the_bits_of_one(cuda, case):
    from paella_amd import ops
    c, k, h, w, (r, s), stride, pad, hint = case
    rng = np.random.default_rng(c * 1000 + k)
    wt, b, x = rnd(rng, k, c, r, s), rnd(rng, k), rnd(rng, 1, c, h, w)
    act = ops.ACT_PRELU if k % 2 else ops.ACT_RELU
    slope = rnd(rng, k) if act == ops.ACT_PRELU else None
    conv = ops.Conv2d(wt, b, stride=stride, pad=pad, act=act, slope=slope, in_hw=(h, w), has_residual=True, tile_hint=hint)
    assert conv.plan.kw == (4 if c % 8 else 8)
    res = rnd(rng, 1, k, conv.plan.P, conv.plan.Q)
    xd, rd = torch.tensor(x, device=cuda), torch.tensor(res, device=cuda)
    conv.plan.small = 0
    want = conv(xd, residual=rd)
    conv.plan.small = 4
    for _ in range(2):  # the second finds the counters of a split reduction as the first left them
        out = torch.full_like(want, float("nan"))
        assert torch.equal(conv(xd, residual=rd, out=out), want)
    # n products and their sum in fp32, each rounded once: an error of at most n * 2^-24 of the sum of their sizes
    ref = reference(x, wt, b, stride, pad, res, slope, int(act))
    size = reference(np.abs(x), np.abs(wt), np.abs(b), stride, pad, np.abs(res), None, 0)
    assert ((out.cpu().double() - ref).abs() <= (c * r * s + 2) * 2.0 ** -24 * size).all()


# workgroups of one tile: 590 and 784, below the rule's line and above it; 777, three rows of tiles; 1600 and 2000, four workgroups of two tiles on the
# fullest compute unit against seven and eight of one
@pytest.mark.parametrize("k, h", [(64, 97), (64, 112), (96, 91), (256, 80), (320, 80)])
def test_a_launch_by_itself_takes_two_tiles_where_it_fills_the_device(cuda, k, h):
    from paella_amd import ops
    rng = np.random.default_rng(h)
    conv = ops.Conv2d(rnd(rng, k, 64, 1, 1), rnd(rng, k), act=ops.ACT_RELU, in_hw=(h, h))
    x = torch.tensor(rnd(rng, 1, 64, h, h), device=cuda)
    assert (conv.plan.dims.grid >= 768) == (h != 97)
    got = conv(x)
    conv.plan.small = 0
    assert torch.equal(got, conv(x))


# C, K, H = W, R, stride: layers that are held together
WIDE = [(64, 64, 56, 3, 1), (64, 96, 41, 3, 1), (128, 160, 28, 1, 1), (64, 32, 50, 3, 1), (256, 256, 14, 3, 1), (64, 192, 33, 1, 1), (96, 65, 40, 1, 1)]
TABLE = [(3, 64, 112, 7, 2), (3, 96, 97, 3, 2), (3, 32, 99, 3, 2), (3, 65, 112, 3, 2), (3, 64, 61, 7, 1)]  # three rows of tiles: one per workgroup
FIVE_ROWS = [(3, 64, 112, 7, 2), (3, 160, 97, 3, 2), (3, 32, 99, 3, 2), (3, 65, 112, 3, 2), (3, 64, 61, 7, 1)]


@pytest.mark.parametrize("layers", [WIDE, TABLE, FIVE_ROWS])
def test_packed_problems_of_two_tiles_report_the_workgroups_of_their_plans(ring, cuda, layers):  # noqa: F811
    lib, h = ring
    from paella_amd import ops
    rng = np.random.default_rng(5)
    cases = []
    for c, k, hw, r, stride in layers:
        conv = ops.Conv2d(rnd(rng, k, c, r, r), rnd(rng, k), stride=stride, pad=r // 2, act=ops.ACT_RELU, in_hw=(hw, hw))
        assert conv.plan.kw == (8 if layers is WIDE else 4)
        x = torch.tensor(rnd(rng, 1, c, hw, hw), device=cuda)
        cases.append((conv, x, conv(x)))
    assert sum(c.plan.dims.grid for c, _, _ in cases if c.plan.d.K > 32) >= 768
    torch.cuda.synchronize()
    batch = lib.paella_ring_batch_size()
    with ops.DirectQueue() as q:
        for flags in (NO_START, 0):  # with start messages: workgroups of one tile
            assert lib.paella_pack_enable(1) == 0
            try:
                outs = []
                for j, (conv, x, want) in enumerate(cases):
                    y = torch.zeros_like(want)
                    conv(x, out=y, stream=q.handle, job_id=(j + 1) | flags, notifier=ctypes.c_void_p(lib.paella_ring_notifier(h, j)))
                    outs.append(y)
                assert lib.paella_pack_flush() == 1
                per = [(c.plan.dims.grid + batch - 1) // batch for c, _, _ in cases]
                total = sum(per) * (1 if flags else 2)
                buf = np.zeros(total, np.uint64)
                assert lib.paella_ring_drain(h, buf.ctypes.data, total, 20.0) == total
                m = decode(buf)
                for j, (conv, _, _) in enumerate(cases):
                    ends = (m["job_id"] == j + 1) & (m["is_start"] == 0)
                    assert m["num"][ends].sum() == conv.plan.dims.grid and ends.sum() == per[j], j
                extra = np.zeros(1, np.uint64)
                assert lib.paella_ring_drain(h, extra.ctypes.data, 1, 0.05) == 0
            finally:
                lib.paella_pack_enable(0)
            torch.cuda.synchronize()
            for y, (_, _, want) in zip(outs, cases):
                assert torch.equal(y, want)


# layers of more than 2048 tiles: two, four and eight waves, the offset table, two tiles per workgroup
@pytest.mark.parametrize("c, k, h, w, r", [(16, 96, 149, 149, 1), (24, 128, 117, 149, 1), (3, 65, 199, 150, 3), (64, 192, 113, 111, 3), (64, 161, 113, 111, 1)])
def test_thousands_of_tiles_give_the_bits_of_larger_ones(cuda, c, k, h, w, r):
    from paella_amd import ops
    rng = np.random.default_rng(k)
    wt, b = rnd(rng, k, c, r, r), rnd(rng, k)
    x = torch.tensor(rnd(rng, 1, c, h, w), device=cuda)
    conv = ops.Conv2d(wt, b, pad=r // 2, act=ops.ACT_RELU, in_hw=(h, w))
    assert (conv.plan.mi, conv.plan.ni) == (1, 1) and conv.plan.dims.grid > 2048
    large = ops.Conv2d(wt, b, pad=r // 2, act=ops.ACT_RELU, in_hw=(h, w), tile_hint=0x120 | (conv.plan.kw.bit_length() - 1))
    assert torch.equal(conv(x), large(x))


def test_packed_problems_with_an_input_transform(ring, cuda):  # noqa: F811
    lib, h = ring
    from paella_amd import ops
    rng = np.random.default_rng(9)
    cases = []
    for c, k, hw, r, act in [(64, 64, 56, 3, ops.ACT_NONE), (128, 160, 28, 1, ops.ACT_RELU), (256, 256, 14, 3, ops.ACT_RELU), (64, 32, 50, 3, ops.ACT_NONE),
                             (64, 65, 41, 1, ops.ACT_RELU), (128, 128, 28, 3, ops.ACT_RELU)]:
        conv = ops.Conv2d(rnd(rng, k, c, r, r), rnd(rng, k), pad=r // 2, act=ops.ACT_RELU, in_hw=(hw, hw))
        assert conv.plan.kw == 8
        x = torch.tensor(rnd(rng, 1, c, hw, hw), device=cuda)
        t = dict(in_scale=torch.tensor(rnd(rng, c), device=cuda), in_shift=torch.tensor(rnd(rng, c), device=cuda), in_act=act)
        cases.append((conv, x, t, conv(x, **t)))
    assert sum(c.plan.dims.grid for c, _, _, _ in cases if c.plan.d.K > 32) >= 768
    torch.cuda.synchronize()
    batch = lib.paella_ring_batch_size()
    with ops.DirectQueue() as q:
        assert lib.paella_pack_enable(1) == 0
        try:
            outs = []
            for j, (conv, x, t, want) in enumerate(cases):
                y = torch.zeros_like(want)
                conv(x, out=y, stream=q.handle, job_id=(j + 1) | NO_START, notifier=ctypes.c_void_p(lib.paella_ring_notifier(h, j)), **t)
                outs.append(y)
            assert lib.paella_pack_flush() == 1
            per = [(c.plan.dims.grid + batch - 1) // batch for c, _, _, _ in cases]
            buf = np.zeros(sum(per), np.uint64)
            assert lib.paella_ring_drain(h, buf.ctypes.data, sum(per), 20.0) == sum(per)
            m = decode(buf)
            for j, (conv, _, _, _) in enumerate(cases):
                assert m["num"][m["job_id"] == j + 1].sum() == conv.plan.dims.grid, j
            extra = np.zeros(1, np.uint64)
            assert lib.paella_ring_drain(h, extra.ctypes.data, 1, 0.05) == 0
        finally:
            lib.paella_pack_enable(0)
        torch.cuda.synchronize()
        for y, (_, _, _, want) in zip(outs, cases):
            assert torch.equal(y, want)


# offset tables of 72 128 and 103 232 bytes, in launches that take workgroups of two tiles by themselves
@pytest.mark.parametrize("c, r", [(1001, 3), (516, 5)])
def test_an_offset_table_of_more_than_64_kb(cuda, c, r):
    from paella_amd import ops
    k, h, w, rows = 64, 100, 128, 3
    rng = np.random.default_rng(c)
    wt, b, x = rnd(rng, k, c, r, r), rnd(rng, k), rnd(rng, 1, c, h, w)
    conv = ops.Conv2d(wt, b, pad=r // 2, act=ops.ACT_RELU, in_hw=(h, w))
    assert conv.plan.dims.lds_bytes > 65536 and conv.plan.dims.grid == 800
    xd = torch.tensor(x, device=cuda)
    got = conv(xd)
    conv.plan.small = 0
    assert torch.equal(got, conv(xd))
    top = x[:, :, :rows + r // 2]  # all that the first rows read; the bound is that of the first test
    ref, size = (reference(*(f(a) for a in (top, wt, b)), 1, r // 2, None, None, act)[:, :, :rows] for f, act in ((np.asarray, 1), (np.abs, 0)))
    assert ((got[:, :, :rows].cpu().double() - ref).abs() <= (c * r * r + 1) * 2.0 ** -24 * size).all()


# one notifier counts a job's workgroups of two tiles (which add two), of one tile and of the pooling operator, in messages of 1, 2, 64 and 128
@pytest.mark.parametrize("batch", [1, 2, 64, 128])
def test_one_notifier_for_workgroups_of_two_tiles_of_one_and_of_pooling(cuda, batch):
    from paella_amd import _abi, ops
    lib, h = _abi.ops(), ctypes.c_void_p()
    assert lib.paella_ring_create_batched(8192, 4, batch, ctypes.byref(h)) == 0
    rng = np.random.default_rng(batch)

    def conv_of(c, k, hw, r):
        conv = ops.Conv2d(rnd(rng, k, c, r, r), rnd(rng, k), pad=r // 2, act=ops.ACT_RELU, in_hw=(hw, hw))
        assert conv.plan.kw == 8
        return conv, torch.tensor(rnd(rng, 1, c, hw, hw), device=cuda)

    jobs = [  # convs, and the map that is pooled
        ([conv_of(64, 64, 40, 3), conv_of(256, 256, 14, 3), conv_of(64, 96, 40, 3)], None),  # a split reduction; three rows of tiles: one per workgroup
        ([conv_of(64, 160, 40, 1), conv_of(64, 32, 40, 3)], torch.tensor(rnd(rng, 1, 64, 40, 40), device=cuda)),
        ([conv_of(64, 128, 56, 3)], torch.tensor(rnd(rng, 1, 64, 39, 40), device=cuda)),
    ]
    want = [[conv(x) for conv, x in convs] + ([ops.pool2d(p, 3, 1, pad=1)] if p is not None else []) for convs, p in jobs]
    grids = [sum(c.plan.dims.grid for c, _ in convs) + (0 if p is None else (p.numel() + 511) // 512) for convs, p in jobs]
    assert sum(c.plan.dims.grid for convs, _ in jobs for c, _ in convs if c.plan.d.K not in (32, 96)) >= 768
    torch.cuda.synchronize()
    try:
        with ops.DirectQueue() as q:
            for flags in (NO_START, NO_START, 0):  # the second finds the counters as the first left them; with start messages: workgroups of one tile
                assert lib.paella_pack_enable(1) == 0
                got = []
                for j, (convs, p) in enumerate(jobs):
                    args = dict(stream=q.handle, job_id=(j + 1) | flags, notifier=ctypes.c_void_p(lib.paella_ring_notifier(h, j)))
                    cs, xs = [c for c, _ in convs], [x for _, x in convs]
                    if p is None:
                        got.append(ops.conv2d_group(cs, xs, **args))
                    else:
                        ys, py = ops.conv2d_group_pool(cs, xs, p, 3, 1, pad=1, **args)
                        got.append(list(ys) + [py])
                assert lib.paella_pack_flush() == 1
                ends = [(g + batch - 1) // batch for g in grids]
                total = sum(ends) * (1 if flags else 2)
                buf = np.zeros(total + 1, np.uint64)
                assert lib.paella_ring_drain(h, buf.ctypes.data, total, 20.0) == total
                assert lib.paella_ring_drain(h, buf.ctypes.data + 8 * total, 1, 0.05) == 0
                m = decode(buf[:total])
                for j, g in enumerate(grids):
                    mine = (m["job_id"] == j + 1) & (m["is_start"] == 0)
                    assert m["num"][mine].sum() == g and mine.sum() == ends[j], (j, flags)
                torch.cuda.synchronize()
                for ys, zs in zip(got, want):
                    assert len(ys) == len(zs) and all(torch.equal(a, b) for a, b in zip(ys, zs))
    finally:
        lib.paella_pack_enable(0)
        lib.paella_ring_destroy(h)
