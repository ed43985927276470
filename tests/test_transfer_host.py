"""The host side of the result transfers (HostLink, sm_transfer.hpp) on the CPU: the HIP calls
and the kernels are played by tests/host/transfer_harness.cpp on host memory, which also knows
the device of every stream, event and allocation.

- other_device: a context's calls work, and give the right values, whatever device is current
  when they are made, as the copies on its stream did that they replace.
- no_allocation: a context's first result allocates nothing (sm_vesicle_radius_noalloc).
- first_buffers: the pinned buffers stay below the length (2 to 3 MiB) from which one takes
  hundreds of microseconds to allocate; and downloads of one chunk, its edge and many.
- troubled_team: a worker that cannot be started leaves a download to the others, and one that
  fails under way ends its workers before what they use (under the address sanitizer).
- behind_work: no host thread is busy while a download waits for the GPU's queued work (the
  processor time of the call; spinning, its workers used 600 ms each).
"""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ROCM = "/opt/rocm/include"


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    if not shutil.which("g++") or not os.path.isdir(os.path.join(ROCM, "hip")):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path_factory.mktemp("transfer") / "transfer_harness")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-D__HIP_PLATFORM_AMD__", "-D__align__(x)=alignas(x)", "-I", os.path.join(ROOT, "softmold_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), "-isystem", ROCM,
                    os.path.join(ROOT, "tests", "host", "transfer_harness.cpp"), "-o", exe, "-lpthread"],
                   check=True)
    return exe


@pytest.mark.parametrize("scenario", ["other_device", "no_allocation", "first_buffers", "troubled_team", "behind_work"])
def test_transfer(harness, scenario):
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0:detect_leaks=0")
    r = subprocess.run([harness, scenario], env=env, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
