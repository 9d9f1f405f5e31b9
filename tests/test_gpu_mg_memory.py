"""Multigrid on a card that is nearly full: the set-up takes what the cycle
cannot do without, and the cycle has the same bits as with every buffer."""
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("prec,left,degree", [("F64", 340, 16), ("F32", 520, 3)])
def test_few_direction_buffers(nbx, dev, degree, prec, left):
    import torch
    # a fine vector of 31 MB in FP64; the cycle's FP32 operands take 157 MB, the coarse levels about 100
    box = nbx.Box.make(7, 20, 20, 20, perturb=0.1, seed=63)
    vector = 20 ** 3 * 512 * (8 if prec == "F64" else 4)

    def cycle(full):
        bp = nbx.BP(box, bpmode=True, precon=nbx.PRECON_MG)
        r = bp.device_array("rhs", bp.fieldOffset).clone()
        z, direct = torch.full_like(r, float("nan")), torch.full_like(r, float("nan"))
        torch.cuda.empty_cache()
        hold = []
        while full and (spare := torch.cuda.mem_get_info()[0] - left * MB) >= 32 * MB:
            hold.append(torch.empty(min(spare, 16 << 30) // (2 * MB) * (2 * MB), dtype=torch.uint8, device=dev))
        free = torch.cuda.mem_get_info()[0]
        bp.mg_setup([7, 3, 1], degree, 4, prec=getattr(nbx, "NBX_" + prec))
        taken = free - torch.cuda.mem_get_info()[0]
        del hold
        torch.cuda.empty_cache()
        bp.mg_apply(r, z)
        bp.mg_use_graph(False)
        bp.mg_apply(r, direct)
        assert torch.equal(z, direct)
        return z, taken

    want, all_buffers = cycle(False)
    got, few = cycle(True)
    assert torch.equal(got, want)
    assert few <= all_buffers - vector, (few, all_buffers)
