"""Three-field PCG on the two sides of the lines between its forms (a thread group
per field, the fields in turn, a workgroup per field), by precision of the
operator: the iterates are the oracle's bit for bit whatever the form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F64, F32, BF16 = 0, 1, 2


@pytest.mark.parametrize("N,dims,bpmode,precs", [
    (3, (16, 16, 11), True, (F64,)), (3, (16, 16, 12), False, (F64,)),    # 3072 elements
    (4, (2, 983, 1), True, (F64,)), (4, (7, 281, 1), False, (F64,)),      # 1967
    (4, (1, 2621, 1), False, (BF16,)), (4, (2, 1311, 1), True, (BF16,)),  # 2622
    (9, (5, 131, 1), False, (BF16,)), (9, (16, 41, 1), False, (BF16,)),   # 656
    (11, (5, 17, 1), False, (F64, F32)), (11, (43, 2, 1), False, (F64, F32)),  # 85, 86
    (13, (3, 1, 1), True, (BF16,)), (13, (2, 1, 1), False, (F64, F32, BF16)), (15, (2, 1, 1), True, (F32, BF16))])
def test_forms_match_oracle(nbx, nbo, dev, N, dims, bpmode, precs):
    import torch
    kw = dict(perturb=0.1, seed=80 + N)
    lam1 = 0.0 if bpmode else 0.3
    bp = nbx.BP(nbx.Box.make(N, *dims, **kw), Nfields=3, bpmode=bpmode, lambda1=lam1, precon=nbx.PRECON_JACOBI)
    ob = nbo.OracleBP(nbo.Box.make(N, *dims, **kw), Nf=3, bpmode=bpmode, lambda1=lam1)
    for prec in precs:
        r = torch.from_numpy(ob.rhs.copy()).to(dev)
        x = torch.zeros_like(r)
        rr, xr = ob.rhs.copy(), np.zeros_like(ob.rhs)
        if prec == F64:
            bp.pcg(r, x, 0.0, 3)
            ob.pcg(rr, xr, 0.0, 3, jacobi=True)
        else:
            bp.pcg_mixed(r, x, 1e-30, 3, prec=nbx.NBX_F32 if prec == F32 else nbx.NBX_BF16, inner_tol=1e-20,
                         max_cycles=1)
            ob.pcg_mixed(rr, xr, 1e-30, 3, prec=prec, inner_tol=1e-20, max_cycles=1, jacobi=True)
        assert np.array_equal(x.cpu().numpy(), xr), prec
