"""Cluster splits at the sizes where their passes change (tiles of 4,096
boundaries, 256 tiles) against the oracle: positions, duplicates and all."""
import numpy as np
import pytest

import oracle as O
from distbvh_amd import CollisionWorld
from helpers import to_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU test needs a GPU"
    return torch


@pytest.mark.parametrize("grid", [None, 4, 1])
@pytest.mark.parametrize("n", [4098, 8192, 8193, 8194, 12289, 50000, 256 * 4096 + 1, 256 * 4096 + 2, 300 * 4096])
def test_cluster_splits(n, grid):
    """grid: places per axis (None: any), so that most codes are equal, or all."""
    rng = np.random.default_rng(n)
    c = rng.random((3, n))
    if grid:
        c = np.floor(c * grid) / grid
    d = np.concatenate([c, np.full((1, n), 1e-3)])
    kd, ce = O.elements_sphere(d)
    for bits, od in ((63, 2), (30, 64), (63, 4096)):
        ref = O.Object(kd, ce, od=od, morton_bits=bits)
        with CollisionWorld(od, morton_bits=bits) as w:
            o = w.create_collision_object()
            o.set_entity_data_sphere(to_cuda(d))
            o.init_broadphase()
            assert np.array_equal(o.splits(), ref.splits.astype(np.uint64)), (bits, od)
