"""Three fields over an element list at the counts where the operator keeps the
factors in registers: each field is the one-field result of the whole mesh at
the listed elements, and the others stay as they were."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,bk,f32", [(2, 1, True), (3, 0, True), (4, 1, True), (5, 0, True), (7, 1, True),
                                      (7, 0, True), (6, 0, False), (8, 0, False), (9, 1, False)])
def test_list_at_the_threshold(nbx, dev, N, bk, f32):
    import torch
    lanes, Np = (N + 1) ** 2, (N + 1) ** 3
    count = (64 * 8192 + lanes - 1) // lanes  # the first that keeps the factors, and one workgroup's remainder more
    count += 1
    E = count + 77
    n = E * Np
    gen = torch.Generator(device=dev).manual_seed(5)
    dt, prec = (torch.float32, nbx.NBX_F32) if f32 else (torch.float64, nbx.NBX_F64)
    r = lambda m: torch.rand(m, generator=gen, device=dev, dtype=dt) - 0.5
    g, D, lam, q = r(7 * n), r(lanes), r(2 * n), r(3 * n)
    el = torch.randperm(E, generator=gen, device=dev)[:count].to(torch.int32)
    out = torch.full_like(q, 7.0)
    nbx.axhelm(N, 3, bk, count, n, g, D, lam, q, out, elementList=el, prec=prec)
    for f in range(3):
        one = torch.empty_like(q[:n])
        nbx.axhelm(N, 1, bk, E, n, g, D, lam, q[f * n:(f + 1) * n].clone(), one, prec=prec)
        want = torch.full_like(one, 7.0).view(E, Np)
        want[el.long()] = one.view(E, Np)[el.long()]
        assert torch.equal(out[f * n:(f + 1) * n], want.view(-1)), f


# element counts one below and at the counts where whole meshes turn from a
# workgroup per field to the kept factors
@pytest.mark.parametrize("N,bk,f32,waves", [(1, 1, False, 32768), (2, 0, False, 16384), (2, 1, True, 1024),
                                            (3, 0, False, 1536), (5, 1, False, 8192), (7, 0, False, 1536),
                                            (8, 1, False, 6144), (9, 1, False, 1536)])
@pytest.mark.parametrize("above", [0, 1])
def test_whole_mesh_at_the_lines(nbx, dev, N, bk, f32, waves, above):
    import torch
    lanes, Np = (N + 1) ** 2, (N + 1) ** 3
    E = (64 * waves + lanes - 1) // lanes - 1 + above
    n = E * Np
    gen = torch.Generator(device=dev).manual_seed(6)
    dt, prec = (torch.float32, nbx.NBX_F32) if f32 else (torch.float64, nbx.NBX_F64)
    r = lambda m: torch.rand(m, generator=gen, device=dev, dtype=dt) - 0.5
    g, D, lam, q = r(7 * n), r(lanes), r(2 * n), r(3 * n)
    out, one = torch.full_like(q, float("nan")), torch.empty_like(q[:n])
    nbx.axhelm(N, 3, bk, E, n, g, D, lam, q, out, prec=prec)
    for f in range(3):
        nbx.axhelm(N, 1, bk, E, n, g, D, lam, q[f * n:(f + 1) * n].clone(), one, prec=prec)
        assert torch.equal(out[f * n:(f + 1) * n], one), f
