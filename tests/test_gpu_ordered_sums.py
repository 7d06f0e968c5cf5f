"""Sums that are rounded in element order, on the GPU: the patch centroids, at
the sizes where the staged chunks end, against the same sums one by one."""
import numpy as np
import pytest

from distbvh_amd import GIVEN, CollisionWorld
from helpers import to_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU test needs a GPU"
    return torch


def _ordered_mean(values):
    """(3,) mean of (3, m) values summed left to right from 0."""
    return np.add.accumulate(values, axis=1)[:, -1] / float(values.shape[1])


@pytest.mark.parametrize("kind", ["sphere", "poly", "snapshot"])
def test_patch_centroids_at_chunk_edges(kind):
    sizes = [1, 0, 15, 16, 17, 32, 255, 1023, 1024, 1025, 2047, 2048, 2049, 3100, 31, 5000]
    n = sum(sizes)
    rng = np.random.default_rng(7)
    c = rng.normal(size=(3, n)) * 10.0 ** rng.integers(-3, 4, size=n) + np.array([[1e3], [-2e3], [0.0]])
    with CollisionWorld(len(sizes)) as w:
        o = w.create_collision_object()
        o.set_patch_offsets(np.cumsum(sizes)[:-1])
        if kind == "sphere":
            o.set_entity_data_sphere(to_cuda(np.concatenate([c, np.full((1, n), 0.5)])), split_algorithm=GIVEN)
        elif kind == "poly":
            o.set_entity_data_poly(to_cuda(c[None]), split_algorithm=GIVEN)
        else:
            kd = np.repeat(rng.normal(size=(n, 13)), 2, axis=1)
            kd[:, 1::2] += 1.0
            o.set_entity_data_snapshot(to_cuda(kd), to_cuda(c.T), split_algorithm=GIVEN)
        got = o.local_patches()
    off = np.concatenate([[0], np.cumsum(sizes)])
    for k, m in enumerate(sizes):
        want = _ordered_mean(c[:, off[k]:off[k + 1]]) if m else np.zeros(3)
        assert got[k]["size"] == m
        assert np.array_equal(got[k]["centroid"], want), (k, m)
