"""Device memory of the library's calls (vcsr_mc_amd/csrc/device_memory.hpp), on the CPU: the header
compiled against a stand-in for the runtime with a card of a few gigabytes
(tests/host/memory_harness.cpp, which says what each check expects)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("memory") / "memory")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-Wall", "-Wno-unused-result",
                        "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        os.path.join(ROOT, "tests", "host", "memory_harness.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("check", [
    "kept_blocks_are_given_back", "unused_blocks_of_the_call_are_given_back", "ranges_are_apart",
    "failed_calls_keep_nothing", "threads"])
def test_device_memory(harness, check):
    r = subprocess.run([harness, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
