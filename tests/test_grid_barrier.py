"""The barrier among k_build's workgroups (sm_sort.hip), read in the gfx950 assembly of this
repository's own source.

One thread of a workgroup releases and arrives for all of it.  Its write-back of the cache
reaches what the other waves wrote only if their memory operations are complete by then, and
a workgroup barrier alone does not wait for them: between a wave's last store or atomic to
global memory and the workgroup barrier before the arrival there has to be a wait for vmcnt(0),
the counter of a wave's outstanding vector memory operations.  Without it the histogram adds of
three waves out of four could arrive after other workgroups had summed the histograms.

Read, not run: a race does not show in a test of results.
"""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(ROOT, "softmold_amd", "csrc")


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    """{name: its instructions} of sm_sort.hip, compiled with the build's device flags."""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    from softmold_amd import build as B

    out = str(tmp_path_factory.mktemp("asm") / "sort.s")
    subprocess.run([HIPCC] + B.DEVICE + B.COMMON + ["--cuda-device-only", "-S", os.path.join(CSRC, "sm_sort.hip"), "-o", out],
                   check=True, capture_output=True)
    funcs, name = {}, None
    for line in open(out):
        if m := re.match(r"(_Z\w+):", line):
            name = m.group(1)
            funcs[name] = []
        elif name and line.startswith("\t") and not line.startswith(("\t.", "\t;")):
            funcs[name].append(line.split(";")[0].strip())
        elif line.startswith(".Lfunc_end"):
            name = None
    return funcs


WRITES = re.compile(r"(global|flat|buffer|scratch)_(store|atomic)|s_swappc|s_setpc")


def test_every_wave_waits_before_its_workgroup_arrives(functions):
    builds = {f: ins for f, ins in functions.items() if "k_build" in f}
    assert len(builds) == 2
    for name, ins in builds.items():
        arrivals = [i for i, x in enumerate(ins) if x.startswith("buffer_wbl2")]
        assert arrivals, name
        for a in arrivals:
            barrier = max(i for i in range(a) if ins[i].startswith("s_barrier"))
            for x in reversed(ins[:barrier]):
                if x.startswith("s_waitcnt") and "vmcnt(0)" in x:
                    break
                assert not WRITES.match(x), f"{name}: '{x}' may be outstanding at the arrival's barrier"
            else:
                pytest.fail(f"{name}: no wait before the arrival's barrier")
