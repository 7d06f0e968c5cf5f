"""Element walks at the sizes where their launch shape changes (queries per
wave, the cross-patch walk's two launches) against the brute-force oracle."""
import numpy as np
import pytest

import oracle as O
from distbvh_amd import CollisionWorld
from helpers import FORMS, sort_pairs, to_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU test needs a GPU"
    return torch


def _spheres(n, rng):
    return np.concatenate([rng.random((3, n)), rng.random((1, n)) * 0.5 / max(1.0, n ** (1 / 3))])


@pytest.mark.parametrize("precision", FORMS)
@pytest.mark.parametrize("n", [1, 3, 5, 63, 65, 4095, 4096, 8191, 8193, 16384, 32767, 65535, 65537, 131071, 131073])
def test_queries_per_wave(n, precision):
    rng = np.random.default_rng(n)
    a, b = _spheres(n, rng), _spheres(300, rng)
    (ka, _), (kb, _) = O.elements_sphere(a), O.elements_sphere(b)
    want = sort_pairs(O.brute_pairs(ka, kb))
    with CollisionWorld(8, precision=precision) as w:
        oa, ob = w.create_collision_object(), w.create_collision_object()
        for o, d in ((oa, a), (ob, b)):
            o.set_entity_data_sphere(to_cuda(d))
            o.init_broadphase()
        oa.broadphase(ob)
        assert np.array_equal(sort_pairs(oa.pairs()), want)
        if n <= 8193:
            oa.self_collision()
            assert np.array_equal(sort_pairs(oa.pairs()), sort_pairs(O.brute_self(ka)))


@pytest.mark.parametrize("precision", FORMS)
@pytest.mark.parametrize("na,nb,every", [(63, 65, 1), (300, 500, 7), (2000, 9000, 40), (9000, 2000, 640),
                                         (14000, 20000, 40)])
def test_cross_patch_uneven(na, nb, every, precision):
    """Two meshes as patches, every `every`-th element of one overlapping all
    of the other: waves of many times the usual visits, and in the largest case
    more left-over subtrees than their list holds (65,536)."""
    from distbvh_amd import GIVEN
    rng = np.random.default_rng(na)
    a, b = _spheres(na, rng), _spheres(nb, rng)
    b[0] += 2.0  # apart but for the big ones
    a[3] *= 0.1
    b[3] *= 0.1
    big = rng.permutation(na)[: max(1, na // every)]
    a[3, big] = 6.0
    with CollisionWorld(2, precision=precision) as w:
        o = w.create_collision_object()
        o.set_patch_offsets([na])
        o.set_entity_data_sphere(to_cuda(np.concatenate([a, b], axis=1)), split_algorithm=GIVEN)
        o.init_broadphase()
        o.self_collision_cross_patch()
        got = sort_pairs(o.pairs())
    want = np.stack([np.repeat(np.sort(big), nb), np.tile(np.arange(na, na + nb), len(big))], axis=1)
    assert np.array_equal(got.astype(np.int64), want)
