"""The two halves of a step with something between them: a change of sort mode, or positions
uploaded again, leaves the step as it is without it; and the rest of a step without a first
half takes the forces at the positions there are."""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


@pytest.mark.parametrize("model,lipids", [("bilayer", 300), ("liposome", 5000)])   # dense and window builds
@pytest.mark.parametrize("start", [0, 1, 2])
def test_halves_with_a_change_between(model, lipids, start):
    d = getattr(sm.Mpd, model)(11, lipids, 3.45).system()
    print(f"case phases {model} {lipids} from mode {start}", flush=True)
    a, b = (sm.Solver.from_system(d) for _ in range(2))
    for s in (a, b):
        s.init_forces()
    a.tune("sort_mode", start)
    for step, to in enumerate((1, 2, 0, 1, 0, 2, 2), 1):
        for s in (a, b):
            s.step_first(step)
        a.tune("sort_mode", to)
        if step % 2:
            a.upload(pos=a.download()[0])
        for s in (a, b):
            s.step_finish(step)
        for x, y in zip(a.download(), b.download()):
            assert np.array_equal(x, y)
    # no first half: the pair force of the same positions, and another kick from it
    pos, vel, _, _ = a.download()
    for s in (a, b):
        s.step_finish(9)   # not a box-move step
        s.step_finish(9)   # not a box-move step
    p, v, acc, _ = a.download()
    assert np.array_equal(p, pos) and not np.array_equal(v, vel) and np.all(np.isfinite(acc))
    for x, y in zip(a.download(), b.download()):
        assert np.array_equal(x, y)
    assert np.array_equal(a.cell_keys(), b.cell_keys())
