"""csrc/copy_back.hpp, the copies of mpqp_regions(), over a stub of the HIP
calls: every byte in its place with and without helping threads, nothing made
inside a call, a call that does not depend on threads that come late, no
thread that outlives the context, errors and missing pinned memory; once as
it is and once under the thread sanitizer."""
import os
import subprocess

import pytest

from conftest import ROOT, TESTS

SOURCE = os.path.join(TESTS, "host", "copy_back_test.cpp")
SCENARIOS = ["copies", "no_staging", "late_helper", "held_up_helper", "failed_copy", "joined", "forked"]


@pytest.fixture(scope="module", params=["plain", "thread"])
def binary(request, tmp_path_factory):
    out = str(tmp_path_factory.mktemp(request.param) / "copy_back_test")
    flags = ["-fsanitize=thread"] if request.param == "thread" else []
    subprocess.run(["g++", "-std=c++17", "-O2", "-g", "-Wall", "-pthread", "-I" + os.path.join(TESTS, "host"), *flags,
                    SOURCE, "-o", out], check=True)
    if flags and subprocess.run([out], capture_output=True, timeout=120).returncode != 2:
        pytest.skip("the thread sanitizer does not start here")  # (without a scenario the program ends with 2)
    return request.param, out


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_scenario(binary, scenario):
    kind, path = binary
    if kind == "thread" and scenario == "forked":
        pytest.skip("the sanitizer does not follow a fork of a process with threads")
    r = subprocess.run([path, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]


def test_blocks_and_threads_are_made_by_warm_up():
    """The first regions call of a process is as fast as the others only if
    neither the pinned blocks nor the threads are made in it."""
    with open(os.path.join(ROOT, "mpqpcudasolver_amd", "csrc", "mpqp_hip.hip")) as f:
        src = f.read()
    body = src[src.index("void ensure_ready()"):]
    body = body[:body.index("\n}\n")]
    for call in ("staging.make(", "copy_threads.make("):
        assert src.count(call) == 1 and call in body, call
