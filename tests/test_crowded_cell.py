"""A system with a cell that always holds more beads than a bucket: its counting builds fall
back, and the context leaves them to the sort.  The trajectory is the incremental re-sort's bit
for bit before, while and after it does, and a context told to count again does so."""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


def _system(seed, crowd):
    """A bilayer with `crowd` immobile beads (type 0) in the corner cell of its box."""
    d = dict(sm.Mpd.bilayer(seed, 500, 3.45).system())
    pos = np.asarray(d["pos"]).reshape(-1, 3)
    rng = np.random.default_rng(seed)
    d["pos"] = np.concatenate([pos, (0.1 + 0.8 * rng.random((crowd, 3))) * d["cutoff"]])
    d["type"] = np.concatenate([d["type"], np.zeros(crowd)]).astype(np.int32)
    d["vel"] = np.concatenate([np.asarray(d["vel"]).reshape(-1, 3), np.zeros((crowd, 3))])
    d["acc"] = None
    d["delta_lxy"] = 0.0
    return d


@pytest.mark.parametrize("replicas", [1, 3])
@pytest.mark.parametrize("crowd", [40, 90])
def test_trajectory_of_a_crowded_cell(replicas, crowd):
    ds = [_system(5 + r, crowd if r == 0 else 0) for r in range(replicas)]
    a, b = (sm.Solver.batch(ds) if replicas > 1 else sm.Solver.from_system(ds[0]) for _ in range(2))
    b.tune("sort_mode", 1)
    print(f"case crowded cell of {crowd}, {replicas} replicas", flush=True)
    for s in (a, b):
        s.init_forces()
    step = 1
    for steps, graph in ((20, 0), (100, 0), (50, 1), (70, 0)):
        for s in (a, b):
            s.tune("graph", graph)
            s.run(step, steps)
        for x, y in zip(a.download(), b.download()):
            assert np.array_equal(x, y)
        step += steps
    assert a.tune_get("sort_count_path") == (1 if crowd <= 64 else 0)
    a.upload(pos=a.download()[0])
    a.tune("sort_mode", 0)
    a.tune("sort_mode", a.tune_get("sort_mode"))
    for s in (a, b):
        s.run(step, 80)
    for x, y in zip(a.download(), b.download()):
        assert np.array_equal(x, y)
