"""The lists a query keeps on the GPU (re-check stripes, the cross-patch walk's
split list): how far they fill, when they grow, and that the pairs are the
expected ones throughout."""
import numpy as np
import pytest

import oracle as O
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


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_cross_patch_replays_fill_the_same_stripes(seed, precision):
    """A captured cross-patch step whose walk leaves subtrees to its second
    launch, most of its re-check candidates in a few of them: 32 waves of large
    spheres, each with its tops at one of 32 heights, over a sheet of small ones
    in blocks at those heights (within a few fp32 ulps of touching, or well
    inside, or missed).  The eager step sized the list, so every replay on the
    same data fits, in whatever order the subtrees are written."""
    from distbvh_amd import GIVEN
    levels, side, size = 32, 64, 64.0
    na, nb = 64 * levels, side * side
    rng = np.random.default_rng(seed)
    g, r, step = np.repeat(np.arange(levels), 64), 0.25 / side, 2.0 ** -5
    big = np.stack([0.5 + 0.02 * g + 0.001 * rng.random(na), 0.5 + 0.001 * rng.random(na), g * step - size,
                    np.full(na, size)])
    gx, gy = np.meshgrid(np.arange(side), np.arange(side))
    level = rng.permutation(levels)[(gy // 8 * 8 + gx // 8) % levels]
    z = level * step + r + 4e-6 * (2.0 * rng.random(gx.shape) - 1.0)
    small = np.stack([(gx + 0.5).reshape(-1) / side, (gy + 0.5).reshape(-1) / side, z.reshape(-1), np.full(nb, r)])
    data = np.concatenate([big, small], axis=1)
    kd, _ = O.elements_sphere(data)
    want = sort_pairs(O.brute_pairs(kd[:na], kd[na:]))
    want[:, 1] += np.uint64(na)
    buf = to_cuda(np.ascontiguousarray(data))
    with CollisionWorld(2, precision=precision) as w:
        o = w.create_collision_object()
        o.set_patch_offsets([na])

        def step_():
            o.set_entity_data_sphere(buf, split_algorithm=GIVEN)
            o.init_broadphase()
            o.self_collision_cross_patch()

        step_()
        assert np.array_equal(sort_pairs(o.pairs()), want)
        # (the blocks at a wave's own height are its candidates)
        assert o.result_stats()["rechecked_pairs"] > na * nb // levels // 2
        with w.capture() as graph:
            step_()
        try:
            for _ in range(40):
                graph.launch()
                assert o.result_count() == len(want)
            assert np.array_equal(sort_pairs(o.pairs()), want)
        finally:
            graph.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_split_list_comes_with_the_first_cross_patch_query(precision):
    """Only a cross-patch query allocates the split list (65,536 entries at
    least).  Its first one leaves earlier graphs launchable, and a cross-patch step
    captured before it walks without a list: same pairs."""
    from distbvh_amd import GIVEN
    rng = np.random.default_rng(7)
    na, nb = 700, 3000
    data = np.concatenate([rng.random((3, na + nb)), rng.random((1, na + nb)) * 0.02])
    data[0, na:] += 2.0  # apart but for every 40th of the first patch
    data[3, :na:40] = 6.0
    (kd, _) = O.elements_sphere(data)
    own = sort_pairs(O.brute_self(kd))
    cross = own[(own[:, 0] < na) & (own[:, 1] >= na)]
    assert 0 < len(cross) < len(own)
    buf = to_cuda(np.ascontiguousarray(data))
    with CollisionWorld(2, precision=precision) as w:
        o = w.create_collision_object()
        o.set_patch_offsets([na])

        def step(query):
            o.set_entity_data_sphere(buf, split_algorithm=GIVEN)
            o.init_broadphase()
            query()

        graphs = []
        try:
            step(o.self_collision)
            assert np.array_equal(sort_pairs(o.pairs()), own)
            for query, want in ((o.self_collision, own), (o.self_collision_cross_patch, cross)):
                with w.capture() as graph:
                    step(query)
                graphs.append((graph, want))
            before = o.device_bytes()
            step(o.self_collision)
            assert o.device_bytes() == before
            step(o.self_collision_cross_patch)
            assert o.device_bytes() == before + 65536 * 8
            assert np.array_equal(sort_pairs(o.pairs()), cross)
            for _ in range(3):
                for graph, want in graphs:
                    graph.launch()
                    assert o.result_count() == len(want)
                    assert np.array_equal(sort_pairs(o.pairs()), want)
        finally:
            for graph, _ in graphs:
                graph.close()
