"""CPU check of the staged host copies' bookkeeping (public_amd/csrc/host_copy.hpp
over a model of the HIP calls it makes): contexts of several devices in one
process, users that come and go while a copy runs, and what is given back."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CASES = ["devices", "events_bounded", "no_events", "events_again", "users_do_not_wait", "given_back", "made_again",
         "given_back_again"]


@pytest.fixture(scope="module")
def results(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host_copy") / "host_copy_check"
    src = os.path.join(ROOT, "tests", "cpp", "host_copy_check.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "tests", "cpp", "hip_model"),
                    src, "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=100).stdout
    return dict(line.split() for line in out.strip().splitlines())


@pytest.mark.parametrize("case", CASES)
def test_staged_copies(results, case):
    assert results[case] == "1"
