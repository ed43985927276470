"""The autotuner's setting, read with tune_get and given to another context by tune, is the
launch shape that was timed: the pair kernels' chunk is one value for the force and for the
energy traversals (a box-move step's force with dU)."""
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]

KNOBS = ("pair_chunk", "pair_variant", "graph", "sort_mode")


def test_tuned_shape_round_trip():
    d = sm.Mpd.bilayer(1234, 400, 3.45).system()
    a, b = (sm.Solver.from_system(d, delta_lxy=0.05, tension=1.0, seed=3) for _ in range(2))
    shape = {k: a.tune_get(k) for k in KNOBS + ("energy_chunk",)}
    assert shape == {k: b.tune_get(k) for k in shape}
    a.init_forces()
    a.run(0, 16)
    a.autotune(64)
    for k in KNOBS:
        b.tune(k, a.tune_get(k))
    for k in shape:
        assert a.tune_get(k) == b.tune_get(k), k
    with pytest.raises(sm.SmError):
        b.tune("energy_chunk", 4)     # read only
