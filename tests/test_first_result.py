"""The first result that a new context gives: sm_vesicle_radius_noalloc before any other
transfer, then every other result, as a context that gave them in another order."""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


@pytest.mark.parametrize("replicas", [1, 5])
def test_noalloc_radius_is_a_contexts_first_result(replicas):
    ds = [sm.Mpd.liposome(k, 300 + 70 * k, 3.45).system() for k in range(replicas)]
    a, b = (sm.Solver.batch(ds) if replicas > 1 else sm.Solver.from_system(ds[0]) for _ in range(2))
    first = a.vesicle_radius(2, noalloc=True)
    want = (b.measure(), b.box(), b.download(), b.param_derivative((2, 3)), b.vesicle_radius(2))
    got = (a.measure(), a.box(), a.download(), a.param_derivative((2, 3)), a.vesicle_radius(2))
    assert np.array_equal(first, want[4]) and np.all(np.isfinite(first))
    for x, y in zip(got[2], want[2]):
        assert np.array_equal(x, y)
    for k in (0, 1, 3, 4):
        assert np.array_equal(got[k], want[k])
