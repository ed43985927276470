"""States on their way between host and device: the chunks of a large download, the
positions' upload and the cell table's reservation when box moves are launched in pieces."""
import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


def _beads(n, seed=3):
    """n free beads of the lipid tables in a large box."""
    m = sm.Mpd.liposome(1, 50, 3.45)
    d = m.system()
    m.close()
    rng = np.random.default_rng(seed)
    d["type"] = rng.integers(2, 4, n).astype(np.int32)
    d["pos"], d["vel"] = rng.uniform(0.0, d["box"], (n, 3)), rng.normal(0.0, 1.7, (n, 3))
    d["chain"], d["chain_const"] = np.zeros((0, 3), np.int32), np.zeros((0, 4))
    return d


# one chunk of 65536 beads, its edges, one bead into the next, the third buffer's turn
@pytest.mark.parametrize("n", [1, 3, 65535, 65536, 65537, 131072, 131073, 200001])
def test_upload_download_round_trip(n):
    d = _beads(n)
    print(f"case transfer {n} beads", flush=True)
    s = sm.Solver.from_system(d)
    rng = np.random.default_rng(n)
    pos, vel, acc = rng.uniform(0.0, d["box"], (n, 3)), rng.normal(0.0, 1.0, (n, 3)), rng.normal(0.0, 9.0, (n, 3))
    s.upload(pos=pos, vel=vel, acc=acc)
    p, v, a, box = s.download()
    assert np.array_equal(p, pos) and np.array_equal(box, d["box"])
    assert np.array_equal(v, vel.astype(np.float32)) and np.array_equal(a, acc.astype(np.float32))
    pos[n // 2, 1] = -1e-9
    with pytest.raises(sm.SmError):
        s.upload(pos=pos)
    assert np.array_equal(s.download()[0], p)     # a refused upload leaves the state
    s.close()


def test_box_moves_in_pieces_equal_one_run():
    """The reservation of cells follows the boxes whether the moves come in one call or many."""
    d = sm.Mpd.bilayer(1234, 400, 3.45).system()
    out = []
    for pieces in (1, 40):
        s = sm.Solver.from_system(d, delta_lxy=0.3, tension=2.0, seed=11)
        s.init_forces()
        for k in range(pieces):
            s.run(1 + k * (320 // pieces), 320 // pieces)
        out.append(s.download() + (s.mc_stats(),))
        s.close()
    for x, y in zip(out[0][:4], out[1][:4]):
        assert np.array_equal(x, y)
    assert out[0][4] == out[1][4] and out[0][4][1] > 0
    assert not np.array_equal(out[0][3], d["box"])


def test_boxes_of_a_batch_and_after_an_upload():
    ds = [sm.Mpd.bilayer(s, 300, 3.45).system() for s in (5, 6, 7)]
    s = sm.Solver.batch(ds)
    assert np.array_equal(s.box(), [d["box"] for d in ds])
    boxes = np.array([d["box"] * f for d, f in zip(ds, (1.0, 1.25, 1.5))])
    s.upload(box=boxes)
    assert np.array_equal(s.box(), boxes)
    s.init_forces()
    s.run(1, 16)
    pos, _, _, box = s.download()
    assert np.array_equal(box, s.box()) and np.all(pos >= 0.0)
    s.close()
