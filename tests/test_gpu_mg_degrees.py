"""Smoothing degrees whose directions are held to the end of the cycle, just
fill the held set, and exceed it before, at and after the coarse correction:
one V-cycle and two applications in a row against the oracle, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("degree", [1, 2, 3, 4, 5, 6, 7, 8, 9, 16])
def test_degree_matches_oracle(nbx, nbo, dev, degree, prec):
    import torch
    kw = dict(perturb=0.1, seed=61)
    bp = nbx.BP(nbx.Box.make(4, 3, 2, 2, **kw), bpmode=True, precon=nbx.PRECON_MG)
    bp.mg_setup([4, 2, 1], degree, 6, prec=prec)
    mg = nbo.OracleMG(nbo.Box.make(4, 3, 2, 2, **kw), [4, 2, 1], degree=degree, coarse_iters=6, bpmode=True,
                      lambda1=0.0, prec=prec)
    want = mg.vcycle(mg.fine.rhs.copy())
    r = torch.tensor(mg.fine.rhs.copy(), device=dev)
    for graph in (True, False, True):
        bp.mg_use_graph(graph)
        z = torch.full_like(r, float("nan"))
        bp.mg_apply(r, z)
        assert np.array_equal(z.cpu().numpy(), want), graph


@pytest.mark.parametrize("orders,dims", [([3, 1], (5, 1, 1)), ([3, 1], (3, 1, 1)), ([4, 1], (3, 1, 1)),
                                         ([7, 3, 1], (3, 1, 1)), ([5, 2, 1], (1, 5, 1))])
@pytest.mark.parametrize("prec", [0, 1])
def test_transfers_of_several_elements_match_oracle(nbx, nbo, dev, orders, dims, prec):
    """Element counts that leave the last transfer workgroup partly idle."""
    import torch
    kw = dict(perturb=0.1, seed=62)
    bp = nbx.BP(nbx.Box.make(orders[0], *dims, **kw), bpmode=True, precon=nbx.PRECON_MG)
    bp.mg_setup(orders, 2, 4, prec=prec)
    mg = nbo.OracleMG(nbo.Box.make(orders[0], *dims, **kw), orders, degree=2, coarse_iters=4, bpmode=True, lambda1=0.0,
                      prec=prec)
    r = torch.tensor(mg.fine.rhs.copy(), device=dev)
    z = torch.full_like(r, float("nan"))
    bp.mg_apply(r, z)
    assert np.array_equal(z.cpu().numpy(), mg.vcycle(mg.fine.rhs.copy()))
