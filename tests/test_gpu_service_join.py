"""Jobs that join a batch of the service while it runs: submitted when the service
reports the long job's row as running, they end before it."""
import time

import pytest

import sqd
from conftest import PUBLISHED

pytestmark = pytest.mark.gpu


def test_jobs_join_while_the_long_job_runs():
    # More1 in rounds of 512 cuboids: some 2,500 rounds, more than 100 ms
    prog = sqd.Program.from_lemma("more1")
    kw = dict(fp32_prefilter=0, dequeue_buffer_size=512)
    ranges = [(100, 101), (104, 105), (3, 4)]
    with sqd.Core(prog, settings=sqd.default_settings(**kw)) as core:
        want = [core.prove_range(a, b)["counts"] for a, b in ranges]
    with sqd.Service(workers=1, batch_jobs=8, fp32_prefilter=0) as svc:
        svc.set_settings(prog, sqd.default_settings(**kw))
        svc.wait(svc.submit(prog, 127, 128))                  # makes the core
        long_job = svc.submit(prog, 0, 128)
        until = time.perf_counter() + 10
        while svc.stats()["rows_running"] == 0 and time.perf_counter() < until:
            pass
        assert svc.stats()["rows_running"] == 1
        ids = [svc.submit(prog, a, b) for a, b in ranges]
        res = [svc.wait(i) for i in ids]
        assert svc.stats()["rows_running"] == 1                # the long job still runs
        first = svc.wait(long_job)
    c = first["counts"]
    assert (c["num_cuboids"], c["num_leaf_cuboids"]) == PUBLISHED["more1"]
    for r, w in zip(res, want):
        assert r["status"] == 0 and r["counts"] == w and r["joined_running"]
        assert r["queued_seconds"] + r["run_seconds"] < first["run_seconds"]
