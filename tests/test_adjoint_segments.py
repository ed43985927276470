"""sm_adjoint keeps up to 256 MiB of step positions whatever checkpoint interval is asked for
and recomputes the segments before the last from checkpoints.  A trajectory that needs two
segments must give the gradient of one kept whole, bit for bit: the recomputed steps are the
same steps.  The sizes put a segment's end on a box move (step 8) and past it, and the
context must come back untouched.
"""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available
from softmold_amd.adjoint import objective

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]

PAIR = (3, 3)


@pytest.mark.parametrize("lipids,segment", [(320000, 8), (280000, 9)])
def test_two_segments_equal_one(lipids, segment):
    m = sm.Mpd.bilayer(7, lipids, 3.45)
    d = m.system()
    m.close()
    d["delta_lxy"], d["tension"] = 0.05, 1.0
    n = len(d["type"])
    S = 12
    assert (256 << 20) // (32 * n) == segment < S
    s = sm.Solver.from_system(d)
    s.init_forces()
    before = s.download()
    print(f"case adjoint {n} beads, segments of {segment}", flush=True)
    J2, g2 = objective(s, PAIR, S, 3)
    J0, none = objective(s, PAIR, S, 3, grad=False)
    print("case adjoint kept whole", flush=True)
    J1, g1 = objective(s, PAIR, S, S)
    assert J1 == J2 == J0 and none is None
    assert np.array_equal(g1, g2) and np.all(np.isfinite(g1)) and np.any(g1 != 0)
    for x, y in zip(before, s.download()):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("asymmetric", [False, True])
@pytest.mark.parametrize("model,lipids", [("bilayer", 300), ("liposome", 2500)])
def test_objective_of_one_step_is_the_measured_energy(model, lipids, asymmetric):
    """The objective's U comes with the pair force, a measurement's from its own traversal: the
    same terms in other orders.  The positions after one step are the same (they follow from the
    initial forces), so J is U_pair + U_chain there, to the roundings of a sum of terms of both
    signs: n_pairs * 2^-53 of the terms' sum, of which U is a good part; 1e-11 is asserted."""
    m = getattr(sm.Mpd, model)(11, lipids, 3.45)
    d = dict(m.system())
    m.close()
    d["delta_lxy"] = 0.0
    if asymmetric:
        f, u = np.array(d["fconst"]), np.array(d["uconst"])
        row = 6 * (2 * d["n_types"] + 3)
        f[row + 1] *= 1.25
        u[row + 1] *= 1.25
        d["fconst"], d["uconst"] = f, u
    s = sm.Solver.from_system(d)
    J, _ = objective(s, PAIR, 1, 1, grad=False)
    s.init_forces()
    s.run(1, 1)
    e = np.asarray(s.measure()).reshape(-1)
    assert J == pytest.approx(e[0] + e[1], rel=1e-11)
