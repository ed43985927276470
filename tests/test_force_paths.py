"""The pair force stages 128 candidates a pass in contexts of 100000 beads and more and 192 in
smaller ones.  A home's candidates are dealt to its lanes by their place in the cell's whole
list, so both must give the same forces bit for bit: a system alone against the same system
beside a filler that takes the context past the line.  The systems hold cells of fewer
candidates than a pass, of several passes, and of more homes than a wave has lanes.
"""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


def _system(n, per_cell, asymmetric, seed):
    """n beads at about per_cell beads a cell of the cutoff's size, a cubic box."""
    m = sm.Mpd.bilayer(7, 30, 3.45)
    d = dict(m.system())
    m.close()
    rng = np.random.default_rng(seed)
    cells = max(3, int(np.ceil((n / per_cell) ** (1 / 3))))
    d["box"] = np.full(3, (cells + 0.3) * d["cutoff"])
    d["pos"] = rng.random((n, 3)) * d["box"]
    d["vel"] = np.zeros((n, 3))
    d["type"] = rng.integers(0, d["n_types"], n).astype(np.int32)
    d["chain"] = np.zeros((0, 3), np.int32)
    d["chain_const"] = np.zeros((0, 4))
    if asymmetric:
        f, u = np.array(d["fconst"]), np.array(d["uconst"])
        row = 6 * (2 * d["n_types"] + 3)
        f[row + 1] *= 1.25
        u[row + 1] *= 1.25
        d["fconst"], d["uconst"] = f, u
    return d


@pytest.mark.parametrize("asymmetric", [False, True])
@pytest.mark.parametrize("n,per_cell", [(1, 1), (700, 4), (3000, 12), (3000, 100)])
def test_both_pass_lengths_give_the_same_forces(n, per_cell, asymmetric):
    print(f"case force paths {n} beads, {per_cell} a cell, asymmetric {asymmetric}", flush=True)
    d, filler = _system(n, per_cell, asymmetric, 3), _system(100000, 3, asymmetric, 4)
    a = sm.Solver.from_system(d)
    b = sm.Solver.batch([d, filler])
    c = sm.Solver.from_system(filler)
    fa, fb, fc = (np.asarray(s.compute_forces()[0]) for s in (a, b, c))
    assert np.array_equal(fb[:n], fa)
    assert np.array_equal(fb[n:], fc)
    assert np.all(np.isfinite(fb)) and (n == 1 or np.any(fa != 0))
    assert np.asarray(a.measure()).reshape(-1)[0] == np.asarray(b.measure()).reshape(2, 3)[0, 0]
