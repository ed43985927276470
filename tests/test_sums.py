"""The device sums of a measurement and of the vesicle radius against numpy at the edges of
their tiles: 512 elements up to 1024 tiles a replica (524288 beads), longer tiles beyond;
replicas without CHAIN molecules; a replica of one bead.

Tolerance: the terms are positive.  A sum passes at most 6 terms a thread (at these sizes),
8 + 8 tree levels and 4 tiles a thread, numpy's at most as many, and a term has fewer than 20
roundings: 64 * 2^-53 each side, 1.5e-14 in all; 1e-13 is asserted.
"""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]

RTOL = 1e-13


def _system(n, chains, seed):
    """n beads anywhere in a box; the first 3 * chains of them are CHAIN molecules of three."""
    m = sm.Mpd.bilayer(7, 30, 3.45)
    d = dict(m.system())
    m.close()
    rng = np.random.default_rng(seed)
    side = max(8.0, 2.0 * np.ceil(n ** (1 / 3)))
    d["box"] = np.array([side, side + 1.0, side + 2.0])
    d["pos"] = rng.random((n, 3)) * d["box"]
    d["vel"] = rng.normal(0.0, 1.7, (n, 3)).astype(np.float32).astype(np.float64)
    d["type"] = rng.integers(2, 4, n).astype(np.int32)
    d["type"][0] = 2
    d["chain"] = np.array([[0, chains, 3]], np.int32) if chains else np.zeros((0, 3), np.int32)
    d["chain_const"] = np.array([[0.7, 100.0, -1.0, 100.0]]) if chains else np.zeros((0, 4))
    return d


def _min_image(d, box):
    d = np.where(d > box / 2, d - box, d)
    return np.where(d < -box / 2, d + box, d)


def _expected(d):
    p, box = d["pos"], d["box"]
    kin = float(((d["vel"] ** 2).sum(1) / 2.0).sum())
    chain = 0.0
    if len(d["chain"]):
        nc = int(d["chain"][0, 1])
        q = p[:3 * nc].reshape(nc, 3, 3)
        a, b = _min_image(q[:, 0] - q[:, 1], box), _min_image(q[:, 1] - q[:, 2], box)
        ra, rb = np.sqrt((a * a).sum(1)), np.sqrt((b * b).sum(1))
        l0, kb, c0, kt = d["chain_const"][0]
        cost = ((a / ra[:, None]) * (b / rb[:, None])).sum(1)
        chain = float((0.5 * kb * ((ra - l0) ** 2 + (rb - l0) ** 2) + 0.5 * kt * (c0 - cost) ** 2).sum())
    h = p[d["type"] == 2]
    x = h - p[0]
    c = (h - np.where(x > box / 2, box, np.where(x < -box / 2, -box, 0.0))).sum(0) / len(h)
    y = h - c
    y = y + np.where(y > box / 2, box, np.where(y < -box / 2, -box, 0.0))
    return chain, kin, float(np.sqrt((y * y).sum(1)).sum() / len(h))


@pytest.mark.parametrize("sizes", [
    [(1, 0)], [(511, 170)], [(512, 0)], [(513, 171)],
    [(1, 0), (3, 1), (1536, 512), (1539, 513), (64, 0)],
    [(524288, 1)], [(524289, 2000)],
], ids=str)
def test_sums_at_tile_edges(sizes):
    print(f"case sums {sizes}", flush=True)
    ds = [_system(n, c, 10 + k) for k, (n, c) in enumerate(sizes)]
    s = sm.Solver.batch(ds) if len(ds) > 1 else sm.Solver.from_system(ds[0])
    for _ in range(2):   # the tickets are back at zero
        m = np.asarray(s.measure()).reshape(len(ds), 3)
        rad = np.asarray(s.vesicle_radius(2)).reshape(len(ds))
        for r, d in enumerate(ds):
            chain, kin, radius = _expected(d)
            assert m[r, 1] == pytest.approx(chain, rel=RTOL)
            assert m[r, 2] == pytest.approx(kin, rel=RTOL)
            assert rad[r] == pytest.approx(radius, rel=RTOL)
    if len(ds) > 1:   # a replica's sums do not depend on the others
        for r, d in enumerate(ds):
            one = sm.Solver.from_system(d)
            assert np.array_equal(np.asarray(one.measure()).reshape(3), m[r])
    s.close()
