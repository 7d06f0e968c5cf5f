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


@pytest.mark.parametrize("precision", FORMS)
def test_batch_with_empty_objects(precision):
    """Batches of growing and shrinking sizes with objects of no element as
    query and as tree, first, between and last: every pair's results, and the
    root boxes of the objects."""
    sizes = [0, 1, 300, 0, 257, 64, 0]
    rng = np.random.default_rng(5)
    data = [(_spheres(max(1, n), rng)[:, :n], _spheres(200, rng)[:, :(0 if n == 64 else 200)])
            for n in sizes]
    with CollisionWorld(4, precision=precision) as w:
        objs = []
        for a, b in data:
            pair = []
            for d in (a, b):
                o = w.create_collision_object()
                o.set_entity_data_sphere(to_cuda(np.ascontiguousarray(d)))
                o.init_broadphase()
                pair.append(o)
            objs.append(pair)
        for take in ([0], [2, 4], [0, 1, 2, 3, 4, 5, 6], [6, 2, 0], [3, 5]):
            w.broadphase_batch([objs[i][0] for i in take], [objs[i][1] for i in take])
            for i in take:
                (ka, _), (kb, _) = O.elements_sphere(data[i][0]), O.elements_sphere(data[i][1])
                want = sort_pairs(O.brute_pairs(ka, kb)) if len(ka) and len(kb) else np.zeros((0, 2), np.uint64)
                assert np.array_equal(sort_pairs(objs[i][0].pairs()), want), (take, i)
        for (a, _), (o, _) in zip(data, objs):
            if a.shape[1]:
                k = O.elements_sphere(a)[0].reshape(-1, 13, 2)
                root = np.asarray(o.root_kdop()).reshape(13, 2)
                assert np.allclose(root[:, 0], k[:, :, 0].min(0), atol=1e-6) and (root[:, 0] <= k[:, :, 0].min(0)).all()
                assert np.allclose(root[:, 1], k[:, :, 1].max(0), atol=1e-6) and (root[:, 1] >= k[:, :, 1].max(0)).all()
