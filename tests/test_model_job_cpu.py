"""Model jobs as they are served, under the real full3 scheduler on the scripted device (the harness takes their launches in the operator
library's place): stages issued several at a time (Context::is_uncrowded, Job::set_stage_span), and instances shared by registrations."""
import numpy as np
import pytest

import _onnx_writer as ow
from _fake import run_harness
from oracle import sched as oracle_sched
from paella_amd import serve

MODEL, KERNELS = "tvm_mobilenet", 54
GROUP = 8


def serve_alone(body, sched="", want=("issued", "lengths"), model=MODEL, **env):
    """`body` with one model type registered, nobody recording stages; the wanted replies as lists."""
    script = "sched full3 streams 8 %s\nrecordlog 0\nclient\njob %s 700000\n" % (sched, serve.job_path(model)) + body
    replies, _ = run_harness(script, PAELLA_STAGE_THREAD="0", **env)
    return [r.split()[1:] for r in replies if r.startswith(want)]


def charge(need):
    """Registers that a launch of these workgroups is charged."""
    blocks, threads, lds, vgprs = (int(v) for v in need.split(","))
    return blocks * oracle_sched.wg_charge(oracle_sched.Stage(False, blocks, threads, lds, vgprs))[0]


def test_a_group_fills_the_entries_of_its_own_stages():
    """From an empty table: one entry per stage after the first request, each an equal share of its group's time."""
    issued, lengths = serve_alone("launch 0 0\ndrain\nissued\nlengths 0\n")
    assert [int(s.rstrip("*")) for s in issued] == list(range(KERNELS))
    ends = [int(s[:-1]) for s in issued if s.endswith("*")]
    assert ends == list(range(GROUP - 1, KERNELS, GROUP)) + [KERNELS - 1]
    assert len(lengths) == 1 + KERNELS  # the input's copy, then the kernels
    for first, last in zip([0] + [e + 1 for e in ends], ends):
        assert len(set(lengths[1 + first:2 + last])) == 1


def test_the_first_stage_is_declared_by_what_is_in_flight_now():
    """A job without an input stage declares kernels as it is made: what an earlier job was told -- few in flight, nobody recording --
    is not what it goes by."""
    alone, recorded, unrecorded = serve_alone("launch 0 0\ndrain\nissued\nprofile on\nlaunch 0 0\ndrain\nissued\nprofile off\nlaunch 0 0\ndrain\nissued\n",
                                              PAELLA_INPUT_RESIDENT="1")
    assert alone[:GROUP] == [str(k) for k in range(GROUP - 1)] + ["%d*" % (GROUP - 1)]
    assert recorded == ["%d*" % k for k in range(KERNELS)]
    assert unrecorded == alone


def test_a_fifth_job_declares_single_stages():
    launches = "".join("launch 0 %d\n" % i for i in range(5))
    first = serve_alone(launches + "issued\ndrain\n", "extra 48", PAELLA_INPUT_RESIDENT="1")[0]
    group = [str(k) for k in range(GROUP - 1)] + ["%d*" % (GROUP - 1)]
    assert first == group * 4 + ["0*"]


def test_a_group_is_charged_as_its_largest_kernel():
    """Registers for two of the first group's last kernel, but not for two of its largest: the second job waits for the first one's
    group, and what that was charged for is given back, so that both are answered (the harness fails otherwise)."""
    needs = serve_alone("launch 0 0\ndrain\nissued\n", want=("needs",), PAELLA_INPUT_RESIDENT="1")[0]
    regs = [charge(need) for need in needs]
    largest, last = max(regs[:GROUP]), regs[GROUP - 1]
    assert 2 * last < largest
    plenty = 1 << 40
    first, rest = serve_alone("launch 0 0\nlaunch 0 1\nissued\ndrain\nissued\n", "extra 0 budget %d %d %d %d" % (largest + last, plenty, plenty, plenty),
                              ("issued",), PAELLA_INPUT_RESIDENT="1")
    assert first == [str(k) for k in range(GROUP - 1)] + ["%d*" % (GROUP - 1)]
    assert len(rest) == 2 * KERNELS - GROUP


def test_idle_instances_are_shared_with_direct_dispatch_only():
    """A second registration of the same library finds the first one's instance; with HIP launches it makes its own."""
    second = "job %s 700000\nlaunch 0 0\ndrain\nlaunch 1 0\ndrain\nlaunch 1 0\ndrain\ninstances\n" % serve.job_path(MODEL)
    assert serve_alone(second, want=("instances",)) == [["1"]]
    assert serve_alone(second, want=("instances",), PAELLA_DISPATCH="hip") == [["2"]]


def conv(b, x, k, c, r=1):
    return b.op("Relu", [b.op("Conv", [x, b.const(b.randn(k, c, r, r, scale=0.1)), b.const(b.randn(k))], kernel_shape=[r, r], pads=[r // 2] * 4)])


def pool(b, x, r):
    return b.op("MaxPool", [x], kernel_shape=[r, r], strides=[r, r])


@pytest.mark.parametrize("limit, want", [
    ("6399", "pooled pooled 4*"),              # the first conv's own 25 workgroups are beyond it: a group of one of few requests, which no limit bounds
    ("6400", "0 1 2 3 4*"), ("8191", "0 1 2 3 4*"), ("8192", "0 1 pooled 4*"), ("12543", "0 1 pooled 4*"),
    ("12544", "pooled pooled 4*"), (None, "pooled pooled 4*"),
])
def test_convs_with_their_pools_keep_to_the_limit_of_small_kernels(limit, want):
    """The small CNN's pairs have 49 workgroups of 256 threads and 16 of 512: beyond the limit they are two launches."""
    env = {} if limit is None else {"PAELLA_GROUP_THREADS": limit}
    issued = serve_alone("launch 0 0\ndrain\nissued\n", want=("issued",), model="tvm_mnist", **env)[0]
    assert issued == want.split()


def test_a_pair_beyond_the_default_limit_is_two_launches(tmp_path):
    """72 workgroups of 512 threads and a small pool, but 256 workgroups as one launch."""
    b = ow.Builder(np.random.default_rng(1))
    y = pool(b, conv(b, "x", 16, 16, 3), 3)
    b.save(str(tmp_path / "mnist-8.onnx"), [("x", [1, 16, 48, 48])], [(y, [1, 16, 16, 16])])
    y = conv(b, y, 16, 16)
    b.save(str(tmp_path / "second.onnx"), [("x", [1, 16, 48, 48])], [(y, [1, 16, 16, 16])])
    issued = serve_alone("launch 0 0\ndrain\nissued\n", want=("issued",), model="tvm_mnist", LLIS_MODELS_DIR=str(tmp_path))[0]
    assert issued == ["0", "1*"]
    (tmp_path / "second.onnx").rename(tmp_path / "mnist-8.onnx")
    for limit, want in (("65536", ["0", "1", "2*"]), ("131072", ["pooled", "2*"])):
        issued = serve_alone("launch 0 0\ndrain\nissued\n", want=("issued",), model="tvm_mnist", LLIS_MODELS_DIR=str(tmp_path), PAELLA_GROUP_THREADS=limit)[0]
        assert issued == want


def test_a_group_is_charged_for_a_pair_as_it_goes_out(tmp_path):
    """The pair has more workgroups than either of its stages: registers for one pair and one of the group's last kernel, and the second job waits."""
    b = ow.Builder(np.random.default_rng(2))
    y = conv(b, pool(b, conv(b, "x", 16, 16, 3), 3), 16, 16)
    b.save(str(tmp_path / "mnist-8.onnx"), [("x", [1, 16, 48, 48])], [(y, [1, 16, 16, 16])])
    env = dict(model="tvm_mnist", LLIS_MODELS_DIR=str(tmp_path), PAELLA_INPUT_RESIDENT="1", PAELLA_GROUP_THREADS="1")
    pair, last = [charge(n) for n in serve_alone("launch 0 0\ndrain\nissued\n", want=("needs",), **env)[0]]
    assert 256 * 512 * 128 == pair > 3 * last
    plenty = 1 << 40
    first, rest = serve_alone("launch 0 0\nlaunch 0 1\nissued\ndrain\nissued\n", "extra 0 budget %d %d %d %d" % (pair + last, plenty, plenty, plenty), ("issued",), **env)
    assert first == rest == ["pooled", "2*"]
