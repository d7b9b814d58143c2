"""Copies of large device arrays into pageable memory (csrc/host_copy.cpp), on
the CPU: the code is linked with a fake HIP runtime (tests/cpp/fake_hip.h)
whose streams can be made to wait."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "hemelb_amd", "csrc")
CPP = os.path.join(ROOT, "tests", "cpp")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_copy") / "check")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Wno-missing-field-initializers",
                    "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", CSRC,
                    "-I", CPP, os.path.join(CSRC, "host_copy.cpp"),
                    os.path.join(CPP, "host_copy_check.cpp"), "-pthread", "-o", exe], check=True)

    def run(scenario):
        r = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
        words = r.stdout.split()
        return dict(zip(words[::2], map(float, words[1::2])))
    return run


def test_a_small_copy_leaves_the_staging_memory_to_others(check):
    # 65 chunks of 1 MiB, all through the staging memory
    assert check("small_beside_large")["staged"] == 65


def test_waiting_for_the_steps_before_it_costs_no_processor_time(check):
    # 0.4 s of waiting, of which a tenth of one processor is allowed
    assert check("waiting")["cpu"] < 0.04


def test_a_copy_that_waits_for_its_steps_leaves_the_staging_memory_to_others(check):
    assert check("large_beside_waiting")["staged"] == 65


def test_the_solvers_device_need_not_be_the_current_one(check):
    assert check("other_device") == {"error": 0, "current": 0, "staged": 65}
