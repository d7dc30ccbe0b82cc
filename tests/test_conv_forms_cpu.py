"""Which kernel a conv's launch takes, and what it asks of the runtime, without a device: tests/fake_device/launch_check.cpp."""
import os
import subprocess

import pytest

from _fake import FAKE_LIB, ensure_built


def launches(*layers):
    """Per layer (route, C, K, H, W, R, S, stride, pad, tile hint, small, flags of the job id, calls): the plan's workgroups, and for each launch
    (kernel, workgroups, dynamic LDS, the most that was asked for)."""
    ensure_built()
    out = subprocess.run([os.path.join(FAKE_LIB, "launch_check")], input="".join(" ".join(map(str, x)) + "\n" for x in layers), capture_output=True,
                         text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    res = []
    for line in out.stdout.splitlines():
        grid, _, rest = line.partition(" ")
        res.append((int(grid), [(a, int(b), int(c), int(d)) for a, b, c, d in (x.split() for x in rest.split(";"))]))
    return res


@pytest.mark.parametrize("c, k, h, w, r", [(1001, 64, 100, 128, 3), (516, 64, 100, 128, 5)])
@pytest.mark.parametrize("route, small", [("alone", -1), ("alone", 4), ("alone", 0), ("packed", -1)])
def test_more_than_64_kb_of_lds_are_asked_for(c, k, h, w, r, route, small):
    """An offset table of a long reduction, in every form that a launch takes."""
    [(_, [(_, _, lds, allowed)])] = launches((route, c, k, h, w, r, r, 1, r // 2, 0, small, 0x80000000, 1))
    assert 65536 < lds <= allowed
