"""The host side of a context (sm_capi.cpp) on the CPU: tests/host/context_harness.cpp stands
in for the HIP runtime and the kernels, with device memory in host memory under the address
sanitizer.

- growth_fails: an upload of a larger box whose allocations fail one after another leaves a
  context that reports an error or works, with every buffer that a kernel would use in place.
- box_and_shapes: an uploaded box sets the launch shapes that follow from the box.
- step_phases: whatever comes between the two halves of a step (another sort mode, another
  table, or no first half at all), a build is launched on keys that were made for it.
- crowded_cells: counting builds that keep falling back are left to the sort.
- creation: the device memory and the clears that making a context takes.
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
    exe = str(tmp_path_factory.mktemp("context") / "context_harness")
    csrc = os.path.join(ROOT, "softmold_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address", "-D__HIP_PLATFORM_AMD__", "-D__align__(x)=alignas(x)",
                    "-Wno-unused-result", "-I", csrc, "-isystem", ROCM, os.path.join(ROOT, "tests", "host", "context_harness.cpp"),
                    os.path.join(csrc, "sm_capi.cpp"), "-o", exe, "-lpthread", "-Wl,--unresolved-symbols=ignore-all"],
                   check=True)
    return exe


@pytest.mark.parametrize("scenario", ["growth_fails", "box_and_shapes", "step_phases", "crowded_cells", "creation"])
def test_context(harness, scenario):
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0:detect_leaks=0")
    r = subprocess.run([harness, scenario], env=env, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
