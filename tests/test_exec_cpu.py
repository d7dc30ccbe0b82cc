"""When the executor records a pass (paella_exec_forward), on the scripted device, and the host's copies: tests/fake_device/exec_check.cpp."""
import os
import subprocess

from _fake import FAKE_LIB, ensure_built


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
