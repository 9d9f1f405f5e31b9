"""The learned step after cycles whose directions outgrow their buffers, so that
the solution takes some of them up before the last step."""
import numpy as np
import pytest

from test_gpu_learned_mg import PRECS, make, random_net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("degree", [1, 4, 5, 8, 9, 16])
def test_learned_cycle_matches_oracle(nbx, nbo, dev, degree, prec):
    import torch
    bp, mg = make(nbx, nbo, (2, 2, 1), PRECS[prec], degree=degree, coarse=4)
    net, W = random_net(nbx, nbo, 5)
    net.attach(bp)
    bp.mg_set_learned(True)
    mg.set_net(W)
    want = mg.vcycle(mg.fine.rhs.copy())
    r = torch.tensor(mg.fine.rhs, device=dev)
    for graph in (True, False, True):
        bp.mg_use_graph(graph)
        z = torch.full_like(r, float("nan"))
        bp.mg_apply(r, z)
        assert np.array_equal(z.cpu().numpy(), want), graph
