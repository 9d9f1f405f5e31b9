"""Parameter gradients at the limits of their arguments: chunks up to the
largest int, and element outputs whose derivative is not finite."""
import numpy as np
import pytest

from test_gpu_net import make, net_with, random_net

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case(nbx, nbo, dev):
    import torch
    bp, ob = make(nbx, nbo, dims=(2, 1, 1))
    rng = np.random.default_rng(11)
    W = nbo.bf16_round(random_net(rng))
    net = net_with(nbx, nbo, bp, W)
    n = bp.fieldOffset
    R = (rng.standard_normal((2, n)) * 1e-2).astype(np.float32)
    Ev = (rng.standard_normal((2, n)) * 1e-1).astype(np.float32)
    net.set_pairs(bp, torch.tensor(R, device=dev), torch.tensor(Ev, device=dev))
    invNorm = np.array([nbo.sumsq_inv_f(e) for e in Ev])
    feat = nbo.net_features(ob.E, 512, ob.mesh["ggeo"])
    samples = np.stack([rng.integers(0, 2, 5), rng.integers(0, 2, 5)], axis=1).astype(np.int32)

    def oracle(s, chunk, G=None):
        return nbo.net_gradient(s, chunk, n, R.ravel(), Ev.ravel(), invNorm, W, feat, ob.invdiag(), G=G)
    return bp, net, samples, n, oracle


@pytest.mark.parametrize("chunk", [5, 6, 2 ** 31 - 5, 2 ** 31 - 1])
def test_chunk_past_the_batch(case, chunk):
    bp, net, samples, _, oracle = case
    g, loss = net.gradient(bp, samples, chunk)
    og, oloss = oracle(samples, 5)
    assert np.array_equal(g, og) and loss == oloss


# a derivative that is not finite reaches the parameters of the taps whose
# neighbour lies in the element, and no others
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 1e43])
@pytest.mark.parametrize("node", [0, 7, 56 + 448, 511, 8 * 3, 64 * 3 + 8 * 4 + 4])
def test_derivative_that_is_not_finite(case, dev, value, node):
    import torch
    bp, net, _, n, oracle = case
    G = np.random.default_rng(node).standard_normal(n)
    G[512 + node] = value
    samples = np.array([[0, 1], [1, 0]], dtype=np.int32)
    g, _ = net.gradient(bp, samples, 16, G=torch.tensor(G, device=dev))
    og, _ = oracle(samples, 16, G=G)
    assert np.isfinite(og).sum() < og.size
    assert np.array_equal(g, og, equal_nan=True)
