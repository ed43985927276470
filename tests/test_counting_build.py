"""The counting build of small cell tables (sort_mode 0 and 2 while the table holds at most
2^18 cells) against the incremental re-sort (sort_mode 1), whose order it must reproduce
bit for bit: equal keys in bead-index order (include/cuda/cell.h:254-260).

The sizes are the edges of its tiles: a scan tile holds 2048 cells (a table of 9/8 of the
grid's cells), the table's limit is 2^18 cells, a key workgroup holds 256 beads and a wave
64.  Beads are drawn anywhere in the box, in one plane of it (long runs of equal keys) and
in a single cell (one run of every bead); a batch has its tables one after another.
"""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


def _system(n, grid, seed):
    m = sm.Mpd.bilayer(7, 30, 3.45)
    d = dict(m.system())
    m.close()
    rng = np.random.default_rng(seed)
    d["box"] = (np.array(grid) - 0.5) * d["cutoff"]
    d["pos"] = rng.random((n, 3)) * d["box"]
    d["vel"] = np.zeros((n, 3))
    d["type"] = rng.integers(2, 4, n).astype(np.int32)
    d["chain"] = np.zeros((0, 3), np.int32)
    d["chain_const"] = np.zeros((0, 4))
    return d


def _places(d, seed):
    rng = np.random.default_rng(seed)
    p = rng.random(d["pos"].shape) * d["box"]
    flat = p.copy()
    flat[:, 2] = 0.3 * d["cutoff"]
    cell = (rng.random(p.shape) * 0.9 + 1.05) * d["cutoff"]
    return p, flat, cell, p[::-1].copy()


@pytest.mark.parametrize("n,grid", [
    (1, (4, 4, 4)), (63, (4, 5, 6)), (257, (4, 4, 4)),
    (1000, (13, 14, 10)), (1000, (13, 12, 12)),      # tables of 2047 and 2106 cells: 1 and 2 scan tiles
    (3000, (16, 16, 16)),
    (3000, (61, 61, 62)),                            # 259539 cells, the last tile partly past the table
    (3000, (62, 62, 61)),                            # 263794 cells: no longer counted in mode 0
])
def test_counting_build_equals_incremental_order(n, grid):
    print(f"case counting build {n} beads {grid} cells", flush=True)
    d = _system(n, grid, 3)
    ss = [sm.Solver.from_system(d) for _ in range(3)]
    for s, mode in zip(ss, (0, 1, 2)):
        s.tune("sort_mode", mode)
    for pos in _places(d, 5):
        out = []
        for s in ss:
            s.upload(pos=pos)
            s.init_forces()
            out.append(s.download())
        for o in out[1:]:
            for x, y in zip(out[0], o):
                assert np.array_equal(x, y)


def test_counting_build_of_a_batch():
    ds = [_system(500, (5, 6, 7), 1), _system(1, (4, 4, 4), 2), _system(2000, (20, 9, 11), 3)]
    a, b = sm.Solver.batch(ds), sm.Solver.batch(ds)
    b.tune("sort_mode", 1)
    for k in range(3):
        for s in (a, b):
            s.init_forces()
            s.run(k, 1)
        for x, y in zip(a.download(), b.download()):
            assert np.array_equal(x, y)
    a.tune("sort_mode", 1)
    for s in (a, b):
        s.run(3, 4)
    for x, y in zip(a.download(), b.download()):
        assert np.array_equal(x, y)
