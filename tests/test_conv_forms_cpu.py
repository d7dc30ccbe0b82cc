"""Which kernel a conv's launch takes, and what it asks of the runtime, without a device: tests/fake_device/launch_check.cpp."""
import os
import subprocess

import pytest

from _fake import FAKE_LIB, ensure_built


def check(layers):
    """A line per layer (route, C, K, H, W, R, S, stride, pad, tile hint, small, flags of the job id, calls)."""
    ensure_built()
    out = subprocess.run([os.path.join(FAKE_LIB, "launch_check")], input="".join(" ".join(map(str, x)) + "\n" for x in layers), capture_output=True,
                         text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    return out.stdout.splitlines()


def launches(*layers):
    """Per layer the plan's workgroups, and for each launch (kernel, workgroups, dynamic LDS, the most that was asked for)."""
    res = []
    for line in check(layers):
        grid, _, rest = line.partition(" ")
        res.append((int(grid), [(a, int(b), int(c), int(d)) for a, b, c, d in (x.split() for x in rest.split(";"))]))
    return res


@pytest.mark.parametrize("c, k, h, w, r", [(1001, 64, 100, 128, 3), (516, 64, 100, 128, 5)])
@pytest.mark.parametrize("route, small", [("alone", -1), ("alone", 4), ("alone", 0), ("packed", -1)])
def test_more_than_64_kb_of_lds_are_asked_for(c, k, h, w, r, route, small):
    """An offset table of a long reduction, in every form that a launch takes."""
    [(_, [(_, _, lds, allowed)])] = launches((route, c, k, h, w, r, r, 1, r // 2, 0, small, 0x80000000, 1))
    assert 65536 < lds <= allowed


ONE, TWO = 1, 2  # tiles per workgroup


def form(launch):
    return TWO if "tall" in launch[0] else ONE


def alone(c, k, h, w, r=1, stride=1):
    return "alone", c, k, h, w, r, r, stride, r // 2, 0, -1, 0, 1


@pytest.mark.parametrize("layer, grid, want", [
    # a matrix-bound reduction: two of twice the work against three on the fullest compute unit, against four, three against five, ...
    (alone(64, 64, 192, 64, 3), 768, ONE), (alone(64, 64, 193, 64, 3), 772, TWO), (alone(64, 64, 256, 64, 3), 1024, TWO), (alone(64, 64, 257, 64, 3), 1028, ONE),
    (alone(64, 64, 320, 64, 3), 1280, ONE), (alone(64, 64, 321, 64, 3), 1284, TWO), (alone(64, 64, 400, 64, 3), 1600, ONE), (alone(64, 64, 576, 64, 3), 2304, ONE),
    (alone(64, 64, 704, 64, 3), 2816, TWO), (alone(64, 64, 784, 64, 3), 3136, TWO),
    # pointwise
    (alone(256, 64, 288, 64), 1152, ONE), (alone(256, 64, 400, 64), 1600, ONE), (alone(256, 64, 576, 64), 2304, TWO),
    # ... of one or two chunks per wave, and a stride
    (alone(64, 64, 192, 64), 768, ONE), (alone(64, 64, 288, 64), 1152, TWO), (alone(128, 64, 400, 64), 1600, TWO), (alone(136, 64, 288, 64), 1152, ONE),
    (alone(64, 64, 576, 128, 3, 2), 1152, TWO),
    # ... whose fourth workgroup per compute unit would run alone, with inputs of 47 and 16 MB; with others beside it; several taps
    (alone(768, 128, 76, 203), 1932, ONE), (alone(512, 256, 38, 203), 1936, TWO), (alone(768, 128, 101, 203), 2564, TWO), (alone(512, 64, 154, 203, 3), 1954, TWO),
    # the offset table, short and long
    (alone(33, 64, 192, 64, 3), 768, ONE), (alone(33, 64, 288, 64, 3), 1152, ONE), (alone(33, 64, 400, 64, 3), 1600, TWO),
    (alone(1001, 64, 192, 64, 3), 768, TWO), (alone(516, 64, 288, 64, 5), 1152, TWO),
    # an odd number of rows
    (alone(96, 96, 91, 91, 3), 777, ONE), (alone(96, 208, 112, 112, 3), 2744, ONE), (alone(64, 160, 77, 64, 3), 770, TWO), (alone(64, 160, 90, 64, 3), 900, ONE),
])
def test_which_launches_take_two_tiles_by_themselves(layer, grid, want):
    [(got, [launch])] = launches(layer)
    assert got == grid and form(launch) == want
    rows = (layer[2] + 31) // 32
    assert launch[1] == (grid if want == ONE else grid // rows * ((rows + 1) // 2))


def held(times, c, k, h, r=1, stride=1, route="packed"):
    return route, c, k, h, h, r, r, stride, r // 2, 0, -1, 0x80000000, times


@pytest.mark.parametrize("layer, grid, want", [
    # an odd number of rows that loses with two tiles, one that gains; even ones, also where the rule for a launch without company says one
    (held(1, 96, 96, 91, 3), 777, ONE), (held(1, 96, 208, 112, 3), 2744, ONE), (held(1, 64, 288, 56, 3), 882, TWO),
    (held(1, 64, 64, 112, 3), 784, TWO), (held(1, 64, 256, 80, 3), 1600, TWO), (held(1, 3, 160, 224, 7, 2), 1960, TWO),
    (held(1, 64, 64, 110, 3), 758, ONE),
    # the same with an input transform
    (held(1, 96, 96, 91, 3, route="transformed"), 777, ONE), (held(1, 96, 208, 112, 3, route="transformed"), 2744, ONE),
    (held(1, 64, 64, 112, 3, route="transformed"), 784, TWO),
])
def test_which_held_launches_of_one_conv_take_two_tiles(layer, grid, want):
    [(got, [launch])] = launches(layer)
    assert got == grid and form(launch) == want


def test_a_held_launch_whose_workgroups_report_their_start_takes_one_tile():
    assert [form(x) for _, [x] in launches(("packed",) + held(1, 64, 64, 112, 3)[1:11] + (0, 1))] == [ONE]


def in_all(n, grid):
    return grid * n + (-grid % 8) * (n - 1)  # a problem's first workgroup is a multiple of eight


@pytest.mark.parametrize("layer, want", [
    # three rows of tiles with several taps, with one; five
    (held(8, 96, 96, 35, 3), ONE), (held(8, 64, 96, 71, 3), ONE), (held(1, 3, 96, 149, 3), ONE), (held(8, 64, 96, 56), TWO), (held(8, 64, 160, 56, 3), TWO),
    (held(8, 64, 96, 56, 3, route="transformed"), ONE), (held(8, 64, 160, 56, 3, route="transformed"), TWO),
    (held(8, 192, 128, 56, route="transformed"), TWO), (held(8, 64, 64, 56, 3, route="transformed"), TWO),
    # in all fewer workgroups than 768, and just as many
    (held(7, 64, 64, 42, 3), TWO), (held(6, 64, 64, 42, 3), ONE),
])
def test_which_convs_take_two_tiles_in_a_launch_of_several(layer, want):
    [(grid, [launch])] = launches(layer)
    rows, n = (layer[2] + 31) // 32, layer[-1]
    assert launch[1] == in_all(n, grid if want == ONE else grid // rows * ((rows + 1) // 2))


@pytest.mark.parametrize("layer, kernel", [
    ((64, 64, 14, 14, 1, 1, 1, 0, 0, -1, 0, 1), "conv_small"), ((64, 64, 56, 56, 3, 3, 1, 1, 0, -1, 0, 1), "conv_mfma"),
    ((64, 64, 112, 112, 3, 3, 1, 1, 0, -1, 0, 1), "conv_tall"),
])
def test_a_launch_that_the_runtime_refuses_is_no_success(layer, kernel):
    """... by itself and of a group of two (which has no form of two tiles), with the error that is also the number 1."""
    [(_, [alone]), (_, [group])] = launches(("alone",) + layer, ("group",) + layer)
    assert alone[0].startswith(kernel) and group[0].startswith(kernel.replace("tall", "mfma") + "_group")
    assert [x.split()[1:] for x in check([("refused",) + layer, ("refused_group",) + layer])] == [["returned", "1"]] * 2


# The layers of tests/test_conv_tall_gpu.py, whose results and message counts are those of either form: which one they compare.
EDGES = [(64, 33, 1, 1, 1, 1, 1, 0, 0x0113), (72, 64, 5, 7, 1, 1, 1, 0, 0x0113), (64, 65, 4, 8, 3, 3, 1, 1, 0), (64, 96, 11, 3, 3, 3, 1, 1, 0x2113),
         (128, 128, 9, 9, 3, 3, 2, 1, 0x1113), (128, 160, 8, 8, 3, 3, 2, 0, 0), (96, 100, 9, 9, 1, 7, 1, 0, 0), (96, 64, 11, 11, 1, 1, 2, 0, 0),
         (512, 128, 7, 7, 3, 3, 1, 1, 0), (3, 64, 31, 33, 7, 7, 2, 3, 0), (5, 65, 9, 11, 3, 3, 1, 1, 0x0112), (3, 96, 13, 13, 5, 5, 1, 2, 0x1112)]


@pytest.mark.parametrize("layer", EDGES)
def test_a_launch_that_is_asked_for_two_tiles_takes_them(layer):
    assert [form(launch) for _, [launch] in launches(("alone",) + layer + (4, 0, 1), ("alone",) + layer + (0, 0, 1))] == [TWO, ONE]


@pytest.mark.parametrize("k, h, want", [(64, 97, ONE), (64, 112, TWO), (96, 91, ONE), (256, 80, TWO), (320, 80, TWO)])
def test_which_of_the_layers_on_the_device_take_two_tiles(k, h, want):
    [(_, [launch])] = launches(alone(64, k, h, h))
    assert form(launch) == want
