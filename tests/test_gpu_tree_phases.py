"""Trees over the sizes where a build gets another phase (128 leaves a chunk,
128 chunks a phase), with equal codes, one-element patches and patches that
end inside chunks, against the brute-force oracle."""
import numpy as np
import pytest

import oracle as O
from distbvh_amd import GIVEN, CollisionWorld
from helpers import FORMS, sort_pairs, to_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU test needs a GPU"
    return torch


@pytest.mark.parametrize("precision", FORMS)
@pytest.mark.parametrize("shape", ["cloud", "line", "nested"])
@pytest.mark.parametrize("n", [127, 128, 129, 255, 257, 16383, 16384, 16385, 50001])
def test_phases(n, shape, precision):
    rng = np.random.default_rng(n + len(shape))
    c = rng.random((3, n))
    if shape == "line":  # equal codes, in runs
        c[1:] = 0.5
        c[0] = np.round(c[0] * 40) / 40
    elif shape == "nested":  # coordinates of every magnitude: chains of one-sided splits
        c *= 2.0 ** -rng.integers(0, 20, n)
    d = np.concatenate([c, np.full((1, n), 1e-4)])
    q = np.concatenate([c[:, :: max(1, n // 200)], np.full((1, len(c[0, :: max(1, n // 200)])), 0.02)])
    (kd, _), (kq, _) = O.elements_sphere(d), O.elements_sphere(q)
    want = sort_pairs(O.brute_pairs(kq, kd))
    cuts = np.sort(np.concatenate([np.minimum([1, 2, 127, 128, 129], n), rng.integers(1, n, 26)]))
    for given in (False, True):
        with CollisionWorld(32 if given else 8, precision=precision) as w:
            a, b = w.create_collision_object(), w.create_collision_object()
            if given:
                a.set_patch_offsets(np.sort(rng.integers(0, q.shape[1], 31)))
                b.set_patch_offsets(cuts)
            for o, x in ((a, q), (b, d)):
                if given:
                    o.set_entity_data_sphere(to_cuda(x), split_algorithm=GIVEN)
                else:
                    o.set_entity_data_sphere(to_cuda(x))
                o.init_broadphase()
            a.broadphase(b)
            assert np.array_equal(sort_pairs(a.pairs()), want)
            if given:
                starts = np.concatenate([[0], cuts, [n]])
                for k, p in enumerate(b.local_patches()):
                    assert p["size"] == starts[k + 1] - starts[k]
                    if p["size"] == 0:
                        continue
                    box, own = p["kdop"].reshape(-1, 2), kd[starts[k]:starts[k + 1]].reshape(-1, 13, 2)
                    assert np.array_equal(box[:, 0], own[:, :, 0].min(0))
                    assert np.array_equal(box[:, 1], own[:, :, 1].max(0))
