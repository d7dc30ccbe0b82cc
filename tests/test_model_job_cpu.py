"""Model jobs as they are served, under the real full3 scheduler on the scripted device (the harness takes their launches in the operator
library's place): stages issued several at a time (Context::is_uncrowded, Job::set_stage_span), and instances shared by registrations."""
from _fake import run_harness
from oracle import sched as oracle_sched
from paella_amd import serve

MODEL, KERNELS = "tvm_mobilenet", 54
GROUP = 8


def serve_alone(body, sched="", want=("issued", "lengths"), **env):
    """`body` with one model type registered, nobody recording stages; the wanted replies as lists."""
    script = "sched full3 streams 8 %s\nrecordlog 0\nclient\njob %s 700000\n" % (sched, serve.job_path(MODEL)) + body
    replies, _ = run_harness(script, PAELLA_STAGE_THREAD="0", **env)
    return [r.split()[1:] for r in replies if r.startswith(want)]


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
    regs = []
    for need in needs:
        blocks, threads, lds, vgprs = (int(v) for v in need.split(","))
        regs.append(blocks * oracle_sched.wg_charge(oracle_sched.Stage(False, blocks, threads, lds, vgprs))[0])
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
