"""Clients that attach one after the other to one server share its idle job instances (RegisteredJob::IdleInstances): every one of
them gets the answers of its own inputs, also where the settings that instances are made under change in between."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_later_clients_reuse_idle_instances_and_get_their_own_answers(cuda, monkeypatch):
    from paella_amd import models, serve
    monkeypatch.setenv("LLIS_MODEL_SEED", "1")
    ex = models.Exec("mnist", seed=1)
    with serve.Server("attach%d" % os.getpid(), "full3", num_streams=8) as srv:
        for seed, pool, zero_copy in [(3, 4, "65536"), (4, 6, "65536"), (5, 6, "0"), (6, 3, "65536")]:
            monkeypatch.setenv("PAELLA_ZERO_COPY_BYTES", zero_copy)
            r = serve.client_run(srv.name, [(serve.job_path("tvm_mnist"), 1.0, pool)], 0.0, pool, 64, seed=seed, verify=2, expected_bytes=2 * 40)
            assert r["mismatches"] == 0 and r["verified_requests"] == (pool - 2) + pool + 64
            answers = r["expected"].view(np.float32).reshape(2, 10)
            for v in range(2):
                ex.set_input(serve.verify_input(seed, 0, v, 784))
                ex.forward()
                np.testing.assert_allclose(answers[v], ex.get_output(), rtol=1e-5, atol=1e-5)
    ex.close()
