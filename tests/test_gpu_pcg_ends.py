"""Where a preconditioned solve ends: no iteration, one, the iteration limit, a
fixed count, an immediate stop and a residual that is not finite, for the two
schedules whose stopping test is apart from the other dots (multigrid tests
before its cycle, the learned preconditioner after its step)."""
import numpy as np
import pytest

from test_gpu_net import make, net_with, random_net

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solvers(nbx, nbo, dev):
    kw = dict(perturb=0.1, seed=71)
    bp = nbx.BP(nbx.Box.make(5, 3, 2, 2, **kw), bpmode=True, precon=nbx.PRECON_MG)
    bp.mg_setup([5, 2, 1], 2, 6, prec=nbx.NBX_F32)
    mg = nbo.OracleMG(nbo.Box.make(5, 3, 2, 2, **kw), [5, 2, 1], degree=2, coarse_iters=6, prec=1)
    bl, ob = make(nbx, nbo)
    W = nbo.bf16_round(random_net(np.random.default_rng(4), scale3=0.05))
    net = net_with(nbx, nbo, bl, W)
    feat = nbo.net_features(ob.E, 512, ob.mesh["ggeo"])
    return {"mg": (bp, mg.fine.rhs, lambda r, x, tol, n: mg.pcg(r, x, tol, n)[0]),
            "learned": (bl, ob.rhs, lambda r, x, tol, n: ob.pcg_learned(r, x, tol, n, W, feat)[0]), "net": net}


@pytest.mark.parametrize("kind", ["mg", "learned"])
@pytest.mark.parametrize("tol,maxit", [(1e-8, 0), (1e-8, 1), (1e-8, 3), (0.0, 0), (0.0, 1), (0.0, 18), (1e-8, 300),
                                       (2.0, 50)])
def test_end_matches_oracle(solvers, dev, kind, tol, maxit):
    import torch
    bp, rhs, oracle = solvers[kind]
    r = torch.tensor(rhs, device=dev)
    x = torch.zeros_like(r)
    st = bp.pcg(r, x, tol, maxit)
    rr, xr = rhs.copy(), np.zeros_like(rhs)
    ost = oracle(rr, xr, tol, maxit)
    assert (st.iterations, st.converged) == (ost.iterations, ost.converged)
    assert st.rdotr0 == ost.rdotr0 and st.rdotr == ost.rdotr
    assert np.array_equal(x.cpu().numpy(), xr) and np.array_equal(r.cpu().numpy(), rr)


@pytest.mark.parametrize("kind", ["mg", "learned"])
def test_zero_right_hand_side_stops_at_once(solvers, dev, kind):
    import torch
    bp, rhs, _ = solvers[kind]
    r = torch.zeros(rhs.size, dtype=torch.float64, device=dev)
    x = torch.zeros_like(r)
    st = bp.pcg(r, x, 1e-8, 20)
    assert st.iterations == 0 and st.converged == 1 and not x.any()


@pytest.mark.parametrize("kind", ["mg", "learned"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_residual_that_is_not_finite_is_an_error(solvers, nbx, dev, kind, value):
    import torch
    bp, rhs, _ = solvers[kind]
    r = torch.tensor(rhs, device=dev)
    r[int(torch.nonzero(r)[7])] = value
    with pytest.raises(nbx.NbxError, match="breakdown"):
        bp.pcg(r, torch.zeros_like(r), 1e-8, 20)
    r = torch.tensor(rhs, device=dev)  # the handle is usable afterwards
    assert bp.pcg(r, torch.zeros_like(r), 1e-8, 300).converged
