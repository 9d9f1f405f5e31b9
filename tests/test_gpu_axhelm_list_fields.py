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
