"""csrc/copy_back.hpp, the copies of mpqp_regions(), over a stub of the HIP
calls: every byte in its place with and without helping threads, nothing made
inside a call, a call that does not depend on threads that come late, no
thread that outlives the context, errors and missing pinned memory; once as
it is and once under the thread sanitizer."""
import os
import subprocess

import pytest

from conftest import TESTS

SOURCE = os.path.join(TESTS, "host", "copy_back_test.cpp")
SCENARIOS = ["copies", "no_staging", "late_helper", "held_up_helper", "failed_copy", "joined", "forked"]


@pytest.fixture(scope="module", params=["plain", "thread"])
def binary(request, tmp_path_factory):
    out = str(tmp_path_factory.mktemp(request.param) / "copy_back_test")
    flags = ["-fsanitize=thread"] if request.param == "thread" else []
    subprocess.run(["g++", "-std=c++17", "-O2", "-g", "-Wall", "-pthread", "-I" + os.path.join(TESTS, "host"), *flags,
                    SOURCE, "-o", out], check=True)
    return request.param, out


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_scenario(binary, scenario):
    kind, path = binary
    if kind == "thread" and scenario == "forked":
        pytest.skip("the sanitizer does not follow a fork of a process with threads")
    r = subprocess.run([path, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
