"""Gather-scatter of one to seven fields (a grid row each), from a few groups to
more than the chip holds at once: pairs, triples, quads and octets in one
list, singletons and excluded nodes between them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [5, 60000, 700000])
@pytest.mark.parametrize("k", [1, 2, 3, 7])
@pytest.mark.parametrize("type_,dtype,op", [("double", np.float64, "add"), ("int", np.int32, "min"),
                                            ("long long int", np.int64, "max"), ("float", np.float32, "mul")])
def test_groups_and_fields(nbx, dev, groups, k, type_, dtype, op):
    import torch
    rng = np.random.default_rng(groups + k)
    size = rng.choice([1, 2, 2, 2, 3, 4, 8], groups)
    ids = np.repeat(np.arange(1, groups + 1), size)
    ids = np.concatenate([ids, np.zeros(17, dtype=np.int64)])
    rng.shuffle(ids)
    n = ids.size
    v = rng.integers(1, 4, (k, n)).astype(dtype)  # exact in every type, whatever the order
    o = nbx.Ogs(ids)
    t = torch.from_numpy(v.copy().reshape(-1)).to(dev)
    o.gather_scatter_many(t, k, n, type_, op)
    got = t.cpu().numpy().reshape(k, n)
    f = {"add": np.add, "min": np.minimum, "max": np.maximum, "mul": np.multiply}[op]
    order = np.argsort(ids, kind="stable")
    order = order[17:]  # id 0 is excluded
    starts = np.concatenate([[0], np.cumsum(np.bincount(ids)[1:])[:-1]])
    for r in range(k):
        want = v[r].copy()
        want[order] = f.reduceat(v[r][order], starts)[ids[order] - 1]
        assert np.array_equal(got[r], want)
