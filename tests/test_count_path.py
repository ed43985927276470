"""Which path a counting build took: counted per cell, or sorted in the fallback of the same
launch.  Both give the order of the incremental re-sort (sort_mode 1), so only the path's
report tells a build that always falls back from one that counts.

The edge is the bucket of a cell, 64 beads: with 64 in one cell the build counts, with 65 it
sorts; in one table and in a batch's, where one replica's crowded cell sends all to the sort.
"""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available
from test_counting_build import _system

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


def _crowd(d, k, seed):
    """k of the system's beads, taken from all over its index range, in one cell; the others
    two a cell at most, away from it."""
    n = len(d["pos"])
    rng = np.random.default_rng(seed)
    grid = (d["box"] / d["cutoff"]).astype(int)
    size = d["box"] / grid
    cells = rng.permutation(np.arange(1, np.prod(grid)))[:(n + 1) // 2].repeat(2)[:n]
    assert len(cells) == n
    crowd = rng.permutation(n)[:k]
    cells[crowd] = 0
    at = np.stack([cells % grid[0], cells // grid[0] % grid[1], cells // (grid[0] * grid[1])], axis=1)
    return (at + 0.1 + 0.8 * rng.random((n, 3))) * size


def _compare(make, ds, crowds, counted):
    """make(ds) in the default mode and in mode 1: the same accelerations, by the path named."""
    a, b = make(ds), make(ds)
    assert a.tune_get("sort_mode") in (0, 2)
    b.tune("sort_mode", 1)
    for k in crowds:
        pos = np.concatenate([_crowd(d, c, 11 + c) for d, c in zip(ds, k)])
        for s in (a, b):
            s.upload(pos=pos)
            s.init_forces()
        for x, y in zip(a.download(), b.download()):
            assert np.array_equal(x, y)
        assert a.tune_get("sort_count_path") == counted(k)
        assert b.tune_get("sort_count_path") == 0
    a.close()
    b.close()


@pytest.mark.parametrize("n,grid,mode", [(100, (4, 5, 6), 0), (1000, (13, 12, 12), 0), (1000, (13, 12, 12), 2),
                                         (20000, (40, 30, 25), 0)])
def test_path_of_one_table(n, grid, mode):
    print(f"case count path {n} beads {grid} cells mode {mode}", flush=True)
    d = _system(n, grid, 3)

    def make(ds):
        s = sm.Solver.from_system(ds[0])
        s.tune("sort_mode", mode)
        return s

    _compare(make, [d], [(2,), (64,), (65,), (64,), (n // 2 if n > 200 else 100,), (0,)], lambda k: int(k[0] <= 64))


def test_path_of_a_batch():
    ds = [_system(500, (8, 9, 7), 1), _system(300, (7, 7, 7), 2), _system(4000, (20, 18, 15), 3)]
    crowds = [(0, 2, 64), (0, 65, 0), (1, 1, 1), (300, 0, 3000), (64, 64, 64)]
    _compare(sm.Solver.batch, ds, crowds, lambda k: int(max(k) <= 64))
