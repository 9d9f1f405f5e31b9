"""Sums of the sample gradients: batches past the count whose gradients are
held at once, chunks that end inside such a batch, begin in one and go on in
the next, or exceed it.  The samples are two, repeated, so the expected sums
are float32 sums of their two gradients in chunk order."""
import numpy as np
import pytest

from test_gpu_net import make, net_with, random_net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsamples,chunk", [(4096, 16), (4097, 16), (4200, 7), (8195, 5000), (4100, 1)])
def test_gradient_sums_across_batches(nbx, nbo, dev, nsamples, chunk):
    import torch
    bp, _ = make(nbx, nbo, dims=(2, 1, 1))
    rng = np.random.default_rng(5)
    net = net_with(nbx, nbo, bp, nbo.bf16_round(random_net(rng)))
    n = bp.fieldOffset
    R = torch.tensor((rng.standard_normal((1, n)) * 1e-2).astype(np.float32), device=dev)
    E = torch.tensor((rng.standard_normal((1, n)) * 1e-1).astype(np.float32), device=dev)
    net.set_pairs(bp, R, E)
    one = [net.gradient(bp, np.array([[0, e]], dtype=np.int32), 1) for e in range(2)]
    which = rng.integers(0, 2, nsamples)
    g, loss = net.gradient(bp, np.stack([np.zeros_like(which), which], axis=1).astype(np.int32), chunk)
    want, wloss = np.zeros_like(g), 0.0
    for c in range(0, nsamples, chunk):
        part, ploss = np.zeros_like(g), 0.0
        for k in which[c:c + chunk]:
            part = part + one[k][0]
            ploss = ploss + one[k][1]
        want = want + part
        wloss = wloss + ploss
    assert np.array_equal(g, want)
    assert loss == wloss
