"""Sums that are rounded in element order, on the GPU: the patch centroids, at
the sizes where the staged chunks end, against the same sums one by one, and
the splitters' split points, at the sizes where blocks of elements end, on
inputs whose order-rounded sum decides where an element goes, against the
oracle's permutations."""
import numpy as np
import pytest

import oracle as O
from distbvh_amd import GEOM_AXIS, GIVEN, ML_GEOM_AXIS, CollisionWorld
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


@pytest.mark.parametrize("kind", ["sphere", "snapshot"])
@pytest.mark.parametrize("od,extra", [(512, 0), (1024, 0), (2048, 0), (2048, 70), (16384, 0)])
def test_centroids_of_many_patches(od, extra, kind):
    """Patches of few elements (four lanes each from 1,024 patches on, while they
    hold at most 64 elements on average), at the sizes where a lane's batches end,
    with large ones side by side, first, last and a block's number of patches apart."""
    rng = np.random.default_rng(od + extra)
    sizes = rng.choice([0, 0, 1, 2, 7, 8, 9, 15, 16, 17, 40], size=od) + extra
    for k, m in {0: 128, 1: 129, 2: 255, 3: 256, 4: 257, 5: 700, od // 16: 130, od // 2: 127, od // 2 + od // 16: 300,
                 od - 2: 2000, od - 1: 129}.items():
        sizes[k] = m
    n = int(sizes.sum())
    c = rng.normal(size=(3, n)) * 10.0 ** rng.integers(-3, 4, size=n) + np.array([[1e3], [-2e3], [0.0]])
    with CollisionWorld(od) as w:
        o = w.create_collision_object()
        o.set_patch_offsets(np.cumsum(sizes)[:-1])
        if kind == "sphere":
            o.set_entity_data_sphere(to_cuda(np.concatenate([c, np.full((1, n), 0.5)])), split_algorithm=GIVEN)
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


def test_packing_time_does_not_follow_the_patches():
    """Packing 16,384 patches of one element takes about as long as 512 patches
    of 32 (25 against 24 us; 56 with a block for each patch)."""
    import time
    n, best = 16384, {512: 1e9, 16384: 1e9}
    data = to_cuda(np.concatenate([np.random.default_rng(1).random((3, n)), np.full((1, n), 0.01)]))
    worlds = {od: CollisionWorld(od) for od in best}
    try:
        objs = {od: w.create_collision_object() for od, w in worlds.items()}
        for od, o in objs.items():
            o.set_patch_offsets(np.arange(1, od) * (n // od))
            o.set_entity_data_sphere(data, split_algorithm=GIVEN)
            o.init_broadphase()
        for _ in range(200):
            for od, o in objs.items():
                t = time.perf_counter()
                o.pack_patches(device=True)
                worlds[od].synchronize()
                best[od] = min(best[od], time.perf_counter() - t)
    finally:
        for w in worlds.values():
            w.close()
    assert best[16384] < 1.5 * best[512], best


def _split_line(kind, n, rng):
    """x of n points whose mean is one of them, so that the rounded sum decides."""
    k = np.arange(n) - (n - 1) // 2
    if kind == "tenths":  # one sign, inexact steps
        x = 1000.0 + 0.1 * k
    elif kind == "negative":
        x = -5.0 + 0.001 * k
    elif kind == "mixed":  # partial sums through zero and many binades
        x = 0.1 * k
    elif kind == "ties":  # steps of a quarter ulp of the sum: halfway cases
        x = 2.0 ** 40 + 2.0 ** -12 * k
    else:  # one huge element first, then small ones against its ulp
        x = 3.0 + rng.integers(0, 8, n) * 0.25
        x[0] = 2.0 ** 52
        return x
    return x if kind == "mixed" else x[rng.permutation(n)]


@pytest.mark.parametrize("ml", [False, True])
@pytest.mark.parametrize("kind", ["tenths", "negative", "mixed", "ties", "huge"])
@pytest.mark.parametrize("n", [1, 2, 3, 511, 512, 513, 1023, 1025, 1537, 4097, 33001])
def test_split_points_at_block_edges(n, kind, ml):
    rng = np.random.default_rng(n)
    d = np.zeros((4, n))
    d[0] = _split_line(kind, n, rng)
    d[1] = 0.25 * rng.integers(0, 3, n)
    d[3] = 0.125
    kd, ce = O.elements_sphere(d)
    od = 8
    idx, sp = O.split_permutations(kd, ce, 3, ml=ml)
    with CollisionWorld(od) as w:
        o = w.create_collision_object()
        o.set_entity_data_sphere(to_cuda(d), split_algorithm=ML_GEOM_AXIS if ml else GEOM_AXIS)
        parts = [o.patch_elements(k) for k in range(od)]
    assert np.array_equal(np.concatenate(parts).astype(np.uint32), idx)
    assert np.array_equal(np.cumsum([len(p) for p in parts])[:-1].astype(np.uint64), sp)
