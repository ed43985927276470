"""How k_build's workgroups wait for each other (sm_sort.hip), read in the gfx950 assembly of
this repository's own source.

One thread of a workgroup releases and arrives for all of it.  Its write-back of the cache
reaches what the other waves wrote only if their memory operations are complete by then, and
a workgroup barrier alone does not wait for them: between a wave's last store or atomic to
global memory and the workgroup barrier before the arrival there has to be a wait for vmcnt(0),
the counter of a wave's outstanding vector memory operations.  Without it the histogram adds of
three waves out of four could arrive after other workgroups had summed the histograms.

The loop over a workgroup's pieces holds barriers, so every lane has to go round it together: a
barrier in a loop within that loop is one that some lanes repeat without the others.

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
def builds(tmp_path_factory):
    """{name: [(instruction, loop depth)]} of k_build's instances, compiled with the build's flags."""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    from softmold_amd import build as B

    out = str(tmp_path_factory.mktemp("asm") / "sort.s")
    subprocess.run([HIPCC] + B.DEVICE + B.COMMON + ["--cuda-device-only", "-S", os.path.join(CSRC, "sm_sort.hip"), "-o", out],
                   check=True, capture_output=True)
    funcs, name, depth = {}, None, 0
    for line in open(out):
        if m := re.match(r"(_Z\w+):", line):
            name, depth = m.group(1), 0
            funcs[name] = []
        elif re.match(r"(\.LBB\w+:|; %bb)", line):      # a block, with the loop that it is in
            m = re.search(r"Depth=(\d+)", line)
            depth = int(m.group(1)) if m else 0
        elif name and (m := re.match(r" *; =>.*Depth=(\d+)", line)):
            depth = int(m.group(1))
        elif name and line.startswith("\t") and not line.startswith(("\t.", "\t;")):
            funcs[name].append((line.split(";")[0].strip(), depth))
        elif line.startswith(".Lfunc_end"):
            name = None
    found = {f: ins for f, ins in funcs.items() if "k_build" in f}
    assert len(found) == 2
    return found


WRITES = re.compile(r"(global|flat|buffer|scratch)_(store|atomic)|s_swappc|s_setpc")


def test_every_wave_waits_before_its_workgroup_arrives(builds):
    for name, code in builds.items():
        ins = [x for x, _ in code]
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


def test_no_barrier_in_an_inner_loop(builds):
    for name, code in builds.items():
        depths = [d for x, d in code if x.startswith("s_barrier")]
        assert len(depths) > 5 and max(depths) == 1, f"{name}: {depths}"
