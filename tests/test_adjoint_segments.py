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
