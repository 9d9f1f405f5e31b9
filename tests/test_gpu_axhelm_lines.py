"""GPU parity of the operator's line form at the edges of its launch shapes:
every order, a single element, element counts that leave idle slots, and both
sides of the lines between the three-field forms (factors kept in registers,
one workgroup per field, one thread group per field).  FP64 and FP32 results
are the oracle's bit for bit: the same fma chains, whatever the split."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def T(dev, a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def operands(nbo, N, E, Nf, dtype):
    n, Np = E * (N + 1) ** 3, (N + 1) ** 3
    f = lambda a: np.ascontiguousarray(a, dtype=dtype)
    return (f(nbo.urand(N, 6, 7 * n)), f(nbo.urand(N, 7, (N + 1) ** 2)),
            f(np.concatenate([1 + 0.5 * nbo.urand(N, 4, n), 0.5 + 0.4 * nbo.urand(N, 5, n)])),
            f(nbo.urand(N, 2, Nf * n)), n, Np)


@pytest.mark.parametrize("N", range(1, 16))
@pytest.mark.parametrize("E", [1, 37])
def test_every_order_matches_oracle(nbx, nbo, dev, N, E):
    """All field counts and forms, whole mesh and element list, FP64 and FP32."""
    import torch
    for dtype, prec in ((np.float64, nbx.NBX_F64), (np.float32, nbx.NBX_F32)):
        for Nf in (1, 3):
            g, D, lam, q, n, Np = operands(nbo, N, E, Nf, dtype)
            dg, dD, dl, dq = (T(dev, a) for a in (g, D, lam, q))
            for bk in (1, 0):
                if dtype == np.float64:
                    ref = nbo.axhelm(N, Nf, bk, E, n, g, D, lam, q)
                else:
                    ref = np.concatenate([nbo.axhelm_f32(N, 1, bk, E, n, g, D, lam, q[f * n:(f + 1) * n].copy())
                                          for f in range(Nf)])
                out = torch.full((Nf * n,), float("nan"), dtype=dq.dtype, device=dev)
                nbx.axhelm(N, Nf, bk, E, n, dg, dD, dl, dq, out, prec=prec)
                assert np.array_equal(out.cpu().numpy(), ref), (dtype, Nf, bk)
                el = np.arange(E - 1, -1, -2, dtype=np.int32)  # every other element, last first
                out.fill_(-7.0)
                nbx.axhelm(N, Nf, bk, el.size, n, dg, dD, dl, dq, out, elementList=T(dev, el), prec=prec)
                want = np.full((Nf, E, Np), -7.0, dtype=dtype)
                want[:, el] = ref.reshape(Nf, E, Np)[:, el]
                assert np.array_equal(out.cpu().numpy(), want.reshape(-1)), (dtype, Nf, bk, "list")


@pytest.mark.parametrize("N,bk,f32", [(3, 1, True), (7, 0, True), (8, 0, False)])
@pytest.mark.parametrize("above", [0, 1])
def test_three_fields_equal_one_field(nbx, nbo, dev, N, bk, f32, above):
    """One element below and at the count where the three-field operator
    turns to the factors kept in registers: each field is the one-field result."""
    import torch
    lanes, Np = (N + 1) ** 2, (N + 1) ** 3
    E = (64 * 8192 + lanes - 1) // lanes - 1 + above
    n = E * Np
    gen = torch.Generator(device=dev).manual_seed(3)
    dt, prec = (torch.float32, nbx.NBX_F32) if f32 else (torch.float64, nbx.NBX_F64)
    r = lambda m: torch.rand(m, generator=gen, device=dev, dtype=dt) - 0.5
    g, D, lam, q = r(7 * n), r(lanes), r(2 * n), r(3 * n)
    out, one = torch.full_like(q, float("nan")), torch.empty_like(q[:n])
    nbx.axhelm(N, 3, bk, E, n, g, D, lam, q, out, prec=prec)
    for f in range(3):
        nbx.axhelm(N, 1, bk, E, n, g, D, lam, q[f * n:(f + 1) * n].clone(), one, prec=prec)
        assert torch.equal(out[f * n:(f + 1) * n], one), f


# element counts below and at the line between the two three-field PCG forms,
# and orders on each side of it at every count
@pytest.mark.parametrize("N,dims", [(3, (16, 16, 15)), (3, (16, 16, 16)), (4, (3, 2, 1)), (6, (2, 1, 1)),
                                    (8, (2, 2, 1)), (9, (3, 1, 1)), (10, (2, 1, 1)), (11, (2, 1, 1)),
                                    (13, (1, 2, 1)), (14, (2, 1, 1)), (15, (1, 2, 1))])
@pytest.mark.parametrize("bpmode", [False, True])
def test_three_field_pcg_matches_oracle(nbx, nbo, dev, N, dims, bpmode):
    import torch
    kw = dict(perturb=0.1, seed=40 + N)
    lam1 = 0.0 if bpmode else 0.3
    bp = nbx.BP(nbx.Box.make(N, *dims, **kw), Nfields=3, bpmode=bpmode, lambda1=lam1, precon=nbx.PRECON_JACOBI)
    ob = nbo.OracleBP(nbo.Box.make(N, *dims, **kw), Nf=3, bpmode=bpmode, lambda1=lam1)
    r = torch.from_numpy(ob.rhs.copy()).to(dev)
    x = torch.zeros_like(r)
    bp.pcg(r, x, 0.0, 5)
    rr, xr = ob.rhs.copy(), np.zeros_like(ob.rhs)
    ob.pcg(rr, xr, 0.0, 5, jacobi=True)
    assert np.array_equal(x.cpu().numpy(), xr)
    assert np.array_equal(r.cpu().numpy(), rr)


# one workgroup per field: element counts on each side of its line, and not a
# multiple of eight (the XCD order pads the grid)
@pytest.mark.parametrize("N,dims", [(9, (5, 17, 3)), (9, (1, 257, 1)), (10, (1, 255, 1)), (10, (16, 16, 1)),
                                    (11, (1, 255, 1)), (11, (1, 257, 1))])
def test_three_field_pcg_per_field_workgroups_match_oracle(nbx, nbo, dev, N, dims):
    import torch
    kw = dict(perturb=0.1, seed=60 + N)
    bp = nbx.BP(nbx.Box.make(N, *dims, **kw), Nfields=3, bpmode=False, lambda1=0.3, precon=nbx.PRECON_JACOBI)
    ob = nbo.OracleBP(nbo.Box.make(N, *dims, **kw), Nf=3, bpmode=False, lambda1=0.3)
    for prec in (nbx.NBX_F64, nbx.NBX_F32):
        r = torch.from_numpy(ob.rhs.copy()).to(dev)
        x = torch.zeros_like(r)
        rr, xr = ob.rhs.copy(), np.zeros_like(ob.rhs)
        if prec == nbx.NBX_F64:
            bp.pcg(r, x, 0.0, 3)
            ob.pcg(rr, xr, 0.0, 3, jacobi=True)
            assert np.array_equal(r.cpu().numpy(), rr)
        else:
            bp.pcg_mixed(r, x, 1e-30, 3, prec=prec, inner_tol=1e-20, max_cycles=1)
            ob.pcg_mixed(rr, xr, 1e-30, 3, prec=1, inner_tol=1e-20, max_cycles=1, jacobi=True)
        assert np.array_equal(x.cpu().numpy(), xr), prec


@pytest.mark.parametrize("N", [7, 9])
@pytest.mark.parametrize("f16", [False, True], ids=["bf16", "fp16"])
def test_matrix_core_fields_at_any_alignment(nbx, dev, N, f16):
    """The matrix-core operator loads node pairs: operands that start at an odd
    element, with an odd field offset, give the bits of the aligned one-field
    call."""
    import torch
    E, Np = 3, (N + 1) ** 3
    n = E * Np
    off = n + 5
    gen = torch.Generator(device=dev).manual_seed(N)
    geo = torch.float32 if f16 else torch.bfloat16
    prec = nbx.NBX_F16 if f16 else nbx.NBX_BF16_MFMA
    r = lambda m, dt=torch.float32: (torch.rand(m, generator=gen, device=dev) - 0.5).to(dt)
    bits = lambda a: a if f16 else a.view(torch.int16)
    at1 = lambda a: torch.cat([a[:1], a])[1:]  # the same values, one element into an allocation
    g, D, lam, q = r(7 * n, geo), r((N + 1) ** 2), r(2 * off, geo), r(3 * off)
    lam1 = torch.cat([lam[:n], lam[off:off + n]])
    for bk in (1, 0):
        out = torch.full((3 * off + 1,), 7.0, device=dev)[1:]
        nbx.axhelm(N, 3, bk, E, off, bits(at1(g)), at1(D), bits(at1(lam)), at1(q), out, prec=prec)
        for f in range(3):
            one = torch.empty(n, device=dev)
            nbx.axhelm(N, 1, bk, E, n, bits(g), D, bits(lam1), q[f * off:f * off + n].clone(), one, prec=prec)
            assert torch.equal(out[f * off:f * off + n], one), (bk, f)
            assert bool((out[f * off + n:(f + 1) * off] == 7.0).all())
