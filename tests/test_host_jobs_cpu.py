"""Host jobs of the upload (csrc/host_jobs.hpp): all are done where the
process may start some threads, one or none more, and none is still running
when a job's error leaves the scope.  No GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("jobs") / "host_jobs")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-o", exe,
                    os.path.join(HERE, "harness", "host_jobs.cpp"), "-ldl"], check=True)
    return lambda *a: subprocess.run([exe, *map(str, a)], capture_output=True, text=True, check=True, timeout=30).stdout


@pytest.mark.parametrize("threads", [0, 1, 2, 4, 9])
def test_jobs_are_done_without_threads(harness, threads):
    assert harness(threads).split() == ["5", str(min(threads, 5))]


@pytest.mark.parametrize("threads,done", [(0, 2), (1, 2), (2, 5), (9, 5)])
def test_a_failing_job_is_reported_after_the_others(harness, threads, done):
    # on the caller's thread the error comes at once, from a thread after all have been started
    assert harness(threads, "fail").split() == [str(done), str(min(threads, 5)), "job", "1"]
