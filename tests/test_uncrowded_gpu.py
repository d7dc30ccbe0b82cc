"""A request among few issues several stages at once (Context::is_uncrowded): the bits of a request whose stages the scheduler issues
one by one, for stage counts below, at and past whole groups of eight, and as the number in flight crosses the limit of four."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,job", [("mnist", "tvm_mnist"), ("resnet18", "tvm_resnet18"), ("squeezenet1_1", "tvm_squeezenet1_1"),
                                      ("mobilenetv2", "tvm_mobilenet"), ("densenet121", "tvm_densenet121"), ("ultraface320", "tvm_ultraface320")])
def test_a_request_in_groups_gives_the_bits_of_one_that_is_recorded_stage_by_stage(cuda, monkeypatch, name, job):
    from paella_amd import models, serve
    monkeypatch.setenv("LLIS_MODEL_SEED", "1")
    in_bytes, out_bytes = models.io_bytes(name)
    x = np.random.default_rng(3).random(in_bytes // 4, dtype=np.float32)
    outs = []
    for log in (True, False):
        with serve.Server("few%d_%d" % (os.getpid(), log), "full3", num_streams=8, event_log=log) as srv:
            for n in (1, 4):
                outs.append(serve.client_single(srv.name, serve.job_path(job), x, out_bytes // 4, n=n)[0])
        if log:  # a recorded request keeps its stages
            ex = models.Exec(name, seed=1)
            stages = 1 if name == "mnist" else ex.num_stages
            ex.close()
            assert srv.event_log().count("\nD ") >= 5 * stages
    for out in outs[1:]:
        np.testing.assert_array_equal(out, outs[0])


@pytest.mark.parametrize("pool", [2, 4, 5, 7])
def test_answers_stay_right_as_requests_come_and_go_around_the_limit(cuda, monkeypatch, pool):
    from paella_amd import serve
    monkeypatch.setenv("LLIS_MODEL_SEED", "1")
    jobs = [(serve.job_path("tvm_resnet18"), 0.6, pool), (serve.job_path("tvm_mobilenet"), 0.4, pool)]
    with serve.Server("few%d_p%d" % (os.getpid(), pool), "full3", num_streams=32) as srv:
        r = serve.client_run(srv.name, jobs, 0.0, pool, 300, seed=pool, verify=2)
        assert r["mismatches"] == 0 and r["all"]["count"] == 300
