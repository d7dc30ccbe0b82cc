"""The conv forms on 16-row tiles (csrc/hip/conv_small.h) at the edges of their tiles, parts and reductions: the bits of the
32 x 32 kernel, and within fp32 rounding of a float64 convolution."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# C, K, H, W, (R, S), stride, pad, tile hint (0: the plan's own choice of waves and splits)
EDGES = [
    (8, 1, 1, 1, (1, 1), 1, 0, 0),            # one pixel, one channel, one chunk
    (8, 15, 3, 5, (1, 1), 1, 0, 0),           # 15 pixels
    (16, 16, 4, 4, (1, 1), 1, 0, 0),          # whole tiles, two chunks
    (24, 33, 17, 1, (1, 1), 1, 0, 0),         # three chunks over four waves: one of them without any
    (40, 17, 5, 7, (3, 3), 1, 1, 0),          # chunks of one pair in two taps (C / 8 odd)
    (8, 31, 6, 6, (5, 5), 1, 2, 0),           # a tap per chunk
    (64, 40, 9, 9, (1, 7), 1, (0, 3), 0),
    (64, 48, 9, 9, (3, 3), 2, 1, 0),          # paired filter columns
    (24, 20, 8, 8, (3, 3), 2, 0, 0),          # paired columns, an odd number of blocks per tap
    (96, 20, 11, 11, (1, 1), 2, 0, 0),        # pointwise with a stride
    (32, 24, 9, 9, (3, 3), 1, 4, 0),          # padding past the filter's reach
    (128, 24, 7, 7, (3, 3), 1, 1, 0x3113),    # eight splits of eight waves: 64 parts
    (104, 24, 6, 6, (1, 1), 1, 0, 0x2113),    # the last split's last waves without a chunk
    (256, 64, 14, 14, (1, 1), 1, 0, 0x0112),  # four waves, sixteen chunks each
]


def rnd(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


def reference(x, w, b, stride, pad, res, slope, act):
    y = torch.nn.functional.conv2d(torch.tensor(x).double(), torch.tensor(w).double(), torch.tensor(b).double(), stride=stride, padding=pad)
    if res is not None:
        y = y + torch.tensor(res).double()
    if act == 1:
        y = y.clamp(min=0)
    elif act == 3:
        y = torch.where(y > 0, y, y * torch.tensor(slope).double().view(1, -1, 1, 1))
    return y


@pytest.mark.parametrize("form", [2, 3])
@pytest.mark.parametrize("case", EDGES)
def test_small_tiles_give_the_bits_of_the_large_tile(cuda, case, form):
    from paella_amd import ops
    c, k, h, w, (r, s), stride, pad, hint = case
    rng = np.random.default_rng(c * 1000 + k)
    wt, b, x = rnd(rng, k, c, r, s), rnd(rng, k), rnd(rng, 1, c, h, w)
    act = ops.ACT_PRELU if k % 2 else ops.ACT_RELU
    slope = rnd(rng, k) if act == ops.ACT_PRELU else None
    conv = ops.Conv2d(wt, b, stride=stride, pad=pad, act=act, slope=slope, in_hw=(h, w), has_residual=True, tile_hint=hint)
    res = rnd(rng, 1, k, conv.plan.P, conv.plan.Q)
    xd, rd = torch.tensor(x, device=cuda), torch.tensor(res, device=cuda)
    conv.plan.small = 0
    want = conv(xd, residual=rd)
    conv.plan.small = form
    for _ in range(2):
        out = torch.full_like(want, float("nan"))
        assert torch.equal(conv(xd, residual=rd, out=out), want)
    ref = reference(x, wt, b, stride, pad, res, slope, int(act))
    assert (want.cpu().double() - ref).norm() <= 1e-5 * ref.norm() + 1e-6


@pytest.mark.parametrize("form", [2, 3])
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("case", [(8, 16, 5, 3, 1), (40, 33, 7, 7, 1), (264, 20, 6, 6, 1), (24, 17, 7, 5, 3), (64, 16, 4, 4, 3)])
def test_small_tiles_with_an_input_transform(cuda, case, act, form):
    from paella_amd import ops
    c, k, h, w, r = case
    rng = np.random.default_rng(c + k)
    conv = ops.Conv2d(rnd(rng, k, c, r, r), rnd(rng, k), pad=r // 2, in_hw=(h, w))
    x = torch.tensor(rnd(rng, 1, c, h, w), device=cuda)
    scale, shift = torch.tensor(rnd(rng, c), device=cuda), torch.tensor(5 * rnd(rng, c), device=cuda)
    conv.plan.small = 0
    want = conv(x, in_scale=scale, in_shift=shift, in_act=act)
    conv.plan.small = form
    assert torch.equal(conv(x, in_scale=scale, in_shift=shift, in_act=act), want)


def test_the_rule_and_a_group_that_follows_it(cuda):
    """A call's convs take the small tiles together or not at all; the pool that rides with them keeps its bits."""
    from paella_amd import ops
    rng = np.random.default_rng(3)
    x = torch.tensor(rnd(rng, 1, 192, 9, 9), device=cuda)
    convs = [ops.Conv2d(rnd(rng, k, 192, 1, 1), rnd(rng, k), act=ops.ACT_RELU, in_hw=(9, 9)) for k in (64, 40, 8)]
    assert all(cv.plan.small == 1 for cv in convs)
    assert ops.Conv2d(rnd(rng, 8, 192, 1, 1), None, in_hw=(9, 9), tile_hint=0x113).plan.small == 0
    for cv in convs:
        cv.plan.small = 0
    want, want_pool = ops.conv2d_group_pool(convs, [x] * 3, x, 3, 1, pad=1)
    for cv in convs:
        cv.plan.small = 1
    got, got_pool = ops.conv2d_group_pool(convs, [x] * 3, x, 3, 1, pad=1)
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and torch.equal(got_pool, want_pool)
    got = ops.conv2d_group(convs, [x] * 3)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
