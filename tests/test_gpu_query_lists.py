"""The lists a query keeps on the GPU (re-check stripes, the cross-patch walk's
split list): how far they fill, when they grow, and that the pairs are the
expected ones throughout."""
import numpy as np
import pytest

from distbvh_amd import CollisionWorld
from helpers import sort_pairs, to_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU test needs a GPU"
    return torch


def _object(w, data):
    o = w.create_collision_object()
    o.set_entity_data_sphere(to_cuda(np.ascontiguousarray(data)))
    o.init_broadphase()
    return o


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1024, 2048, 4096])
def test_batch_fills_every_stripe(n, precision):
    """Queries of 16 to 64 waves with 768 candidates a wave: a stripe of the
    first list (1,024 entries) holds those of one wave and not of two, so the
    lists stay as they are only if no two waves of a query share a stripe."""
    k, copies = 8, 12
    i = np.arange(n)
    sites = np.stack([i % 16, i // 16 % 16, i // 256]).astype(np.float64)
    rng = np.random.default_rng(n)
    with CollisionWorld(4, precision=precision) as w:
        qs = [_object(w, np.concatenate([sites, np.full((1, n), 0.2)])) for _ in range(k)]
        far = _object(w, np.concatenate([sites + 100.0, np.full((1, n), 0.2)]))
        at = np.tile(sites, copies) + 0.01 * rng.random((3, copies * n))
        near = _object(w, np.concatenate([at, np.full((1, copies * n), 0.2)]))
        w.broadphase_batch(qs, [far] * k)  # (the lists at their first sizes)
        before = [o.device_bytes() for o in qs]
        w.broadphase_batch(qs, [near] * k)
        after = [o.device_bytes() for o in qs]  # (before result_stats, which allocates its own word)
        want = sort_pairs(np.stack([np.tile(i, copies), np.arange(copies * n)], axis=1).astype(np.uint64))
        for o in qs:
            assert o.result_stats()["rechecked_pairs"] == copies * n
            assert np.array_equal(sort_pairs(o.pairs()), want)
        assert after == before
