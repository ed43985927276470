"""An objective without its gradient keeps no positions: its memory does not grow with the
steps or the checkpoint interval, and its value is the one that comes with the gradient."""
import pytest

import softmold_amd as sm
from conftest import gpu_available
from softmold_amd.adjoint import objective

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]


@pytest.mark.parametrize("checkpoint", [1, 200])
def test_objective_alone_keeps_two_buffers(checkpoint):
    """200 steps of 60k beads: 388 MB of positions if all were kept, 3.8 MB in two buffers; the
    context keeps its workspace (up to 512 MiB) after the call, where it is seen."""
    import torch

    m = sm.Mpd.bilayer(7, 20000, 3.45)
    d = m.system()
    m.close()
    d["delta_lxy"], d["tension"] = 0.05, 1.0
    n = len(d["type"])
    print(f"case objective of {n} beads, checkpoint {checkpoint}", flush=True)
    s, t = sm.Solver.from_system(d), sm.Solver.from_system(d)
    for x in (s, t):
        x.init_forces()
        x.run(0, 8)
        x.sync()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    J, g = objective(s, (3, 3), 200, checkpoint, grad=False)
    used = free - torch.cuda.mem_get_info()[0]
    assert g is None and used < 64 << 20, f"{used >> 20} MiB"
    assert objective(t, (3, 3), 200, checkpoint)[0] == J
