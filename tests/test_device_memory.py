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
    "kept_blocks_are_given_back", "unused_blocks_of_the_call_are_given_back", "available_counts_idle_memory",
    "large_reserves_need_room", "blocks_age_by_calls",
    "kept_memory_is_bounded", "ranges_are_apart", "failed_calls_keep_nothing", "threads"])
def test_device_memory(harness, check):
    r = subprocess.run([harness, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_release_without_gpu():
    """With nothing kept the release call does nothing."""
    import vcsr_mc_amd as vm
    vm.release_scratch()


@pytest.mark.gpu
def test_release_gives_memory_back():
    """What a build leaves for later ones is free again after the call, and a format built before it
    is untouched."""
    import numpy as np
    import torch

    import vcsr_mc_amd as vm
    from gpu_util import dev, say
    say("release")
    A = vm.generate(1, 100000)
    B = torch.ones((A.N, 8), device="cuda")
    C = torch.zeros((A.M, 8), device="cuda")
    with vm.DeviceFormat.from_device_csr(dev(A.row_ptr), dev(A.col), dev(A.val), A.M, A.N, True,
                                         32) as f:
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        vm.release_scratch()
        assert torch.cuda.mem_get_info()[0] - before >= 64 * A.nnz
        f.spmm(B, C)
        torch.cuda.synchronize()
    want = np.add.reduceat(np.append(A.val.astype(np.float64), 0.0), A.row_ptr[:-1])
    want[np.diff(A.row_ptr) == 0] = 0.0
    assert np.allclose(C[:, 0].cpu().numpy(), want, rtol=1e-5, atol=1e-5)
