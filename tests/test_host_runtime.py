"""The library's host code against a HIP runtime on the host
(tests/native/fake_hip.hpp): what it asks of the runtime and what it does when a
call fails.  No GPU is used; kernels do not run."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "c-saw_amd", "lib")
ROCM = "/opt/rocm"


@pytest.fixture(scope="module")
def host_check(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(f"{ROCM}/include"):
        pytest.skip("needs g++ and HIP headers")
    exe = str(tmp_path_factory.mktemp("host") / "host_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", "-rdynamic", "-w",
                    os.path.join(HERE, "native", "host_check.cpp"), "-o", exe, f"-L{LIB}", "-lcsaw",
                    f"-Wl,-rpath,{LIB}", f"-Wl,-rpath-link,{ROCM}/lib"], check=True, capture_output=True, timeout=240)
    return exe


def run(exe, name):
    r = subprocess.run([exe, name], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stdout + r.stderr


def test_hub_positions_past_32_bits(host_check):
    run(host_check, "hub_positions")


def test_unwaited_plan_waits_on_its_own_device(host_check):
    run(host_check, "wait_on_own_device")


def test_nothing_is_pooled_after_a_failed_wait(host_check):
    run(host_check, "failed_wait")


def test_calls_that_fail_before_they_have_waited(host_check):
    run(host_check, "failed_copy_out")


def test_partly_made_streams_are_completed(host_check):
    run(host_check, "partial_streams")


def test_pooled_memory_makes_room_for_any_allocation(host_check):
    run(host_check, "pool_makes_room")


def test_narrow_hubs_for_the_plans_that_read_them(host_check):
    run(host_check, "narrow_hubs_when_read")


def test_autotune_tries_what_the_hops_read(host_check):
    run(host_check, "autotune_reads")
