"""Builds of few elements (one launch up to the tree stage) against the oracle:
bounds, sorted codes and permutation, splits, patches and pairs at the sizes
where the launch's shapes end, for every element kind, code width and form."""
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


def _elements(kind, n, rng):
    c = rng.random((3, n))
    c[:, : n // 3] = np.round(c[:, : n // 3] * 4) / 4  # shared places: equal codes
    if kind == "flat":
        c[2] = 0.5  # a degenerate axis
    size = 0.4 / max(1.0, n ** (1 / 3))
    if kind == "sphere":
        return np.concatenate([c, np.full((1, n), size)])
    nv = {"tri": 3, "flat": 3, "hex": 8, "point": 1}[kind]
    off = size * (rng.random((nv, 3, n)) - 0.5)
    if kind == "flat":
        off[:, 2] = 0.0
    return c[None] + off


@pytest.mark.parametrize("kind", ["tri", "flat", "hex", "point", "sphere", "snapshot"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2049, 4095, 4096, 4097, 8193])
def test_small_build_matches_oracle(n, kind):
    rng = np.random.default_rng(n * 7 + len(kind))
    base = "tri" if kind == "snapshot" else kind
    data, other = _elements(base, n, rng), _elements(base, 200, rng)
    eps = 0.01
    elems = O.elements_sphere if kind == "sphere" else lambda d: O.elements_poly(d, eps)
    (kd, ce), (kb, cb) = elems(data), elems(other)
    form = FORMS[n % 3]
    want, want_own = sort_pairs(O.brute_pairs(kd, kb)), sort_pairs(O.brute_self(kd))

    def fill(o, d, k, c):
        if kind == "sphere":
            o.set_entity_data_sphere(to_cuda(d))
        elif kind == "snapshot":
            o.set_entity_data_snapshot(to_cuda(k), to_cuda(c))
        else:
            o.set_entity_data_poly(to_cuda(d), epsilon=eps)
        o.init_broadphase()

    for bits, od in ((63, 1), (63, 16), (30, 4), (63, 2048), (30, 512)):
        ref = O.Object(kd, ce, od=od, morton_bits=bits)
        with CollisionWorld(od, morton_bits=bits, precision=form) as w:
            a, b = w.create_collision_object(), w.create_collision_object()
            fill(a, data, kd, ce)
            fill(b, other, kb, cb)
            a.broadphase(b)
            pairs = sort_pairs(a.pairs())
            codes, perm = a.sorted()
            splits, tree, mn = a.splits(), a.tree(), a.bounds()[0]
            sizes = [p["size"] for p in a.local_patches()] if od <= 16 else None
            a.self_collision()
            own = sort_pairs(a.pairs())
        assert np.array_equal(codes, ref.codes) and np.array_equal(perm, ref.perm), (bits, od)
        assert np.array_equal(splits, ref.splits.astype(np.uint64)), (bits, od)
        assert np.array_equal(mn, kd[:, 0:6:2].min(axis=0))
        if sizes is not None:
            assert sizes == [int(e - s) for s, e in zip(ref.pbegin, ref.pend)]
        assert np.array_equal(pairs, want), (bits, od)
        assert np.array_equal(own, want_own), (bits, od)
        assert tree["root"] < max(1, 2 * n - 1)


@pytest.mark.parametrize("od", [1024, 2048, 4096, 16384])
def test_small_build_of_many_patches(od):
    """fp64 records: the patch slabs of a build of few elements in many patches
    (mostly empty), cleared inside the one launch up to 2,048 patches and by a
    launch of their own above, over those of an earlier build."""
    rng = np.random.default_rng(od)
    with CollisionWorld(od, precision="fp64_records") as w:
        a, b = w.create_collision_object(), w.create_collision_object()
        for n in (900, 1, 700):
            refs = []
            for o in (a, b):
                data = _elements("sphere", n, rng)
                o.set_entity_data_sphere(to_cuda(data))
                o.init_broadphase()
                refs.append(O.Object(*O.elements_sphere(data), od=od))
            a.broadphase(b)
            assert np.array_equal(sort_pairs(a.pairs()), sort_pairs(O.brute_pairs(refs[0].kdops, refs[1].kdops)))
            for o, ref in zip((a, b), refs):
                got = o.local_patches()
                size = (ref.pend - ref.pbegin).astype(np.int64)
                assert [p["size"] for p in got] == size.tolist()
                full = np.nonzero(size)[0]
                assert np.array_equal(np.stack([got[k]["kdop"] for k in full]), ref.patch_kdops[full])
            full_a, full_b = (np.nonzero(r.pend > r.pbegin)[0] for r in refs)
            want = O.brute_pairs(refs[0].patch_kdops[full_a], refs[1].patch_kdops[full_b]).astype(np.int64)
            pairs = sort_pairs(a.patch_pairs())
            assert np.array_equal(pairs.astype(np.int64), np.stack([full_a[want[:, 0]], full_b[want[:, 1]]], axis=1))


def test_small_build_time_does_not_follow_the_patches():
    """The clearing of 16,384 patches' slabs (3.4 MB) is not one workgroup's: a
    build of one element takes about as long as with 64 patches (87 against 85 us;
    126 when one workgroup cleared them)."""
    import time
    best = {64: 1e9, 16384: 1e9}
    data = to_cuda(np.array([[0.1], [0.2], [0.3], [0.05]]))
    worlds = {od: CollisionWorld(od, precision="fp64_records") for od in best}
    try:
        objs = {od: w.create_collision_object() for od, w in worlds.items()}
        for _ in range(200):
            for od, w in worlds.items():
                t = time.perf_counter()
                objs[od].set_entity_data_sphere(data)
                objs[od].init_broadphase()
                w.synchronize()
                best[od] = min(best[od], time.perf_counter() - t)
    finally:
        for w in worlds.values():
            w.close()
    assert best[16384] < 1.3 * best[64], best


@pytest.mark.parametrize("kind", ["tri", "point", "sphere"])
@pytest.mark.parametrize("n", [65, 1500, 4096])
def test_small_build_with_non_finite_coordinates(n, kind):
    """Elements with NaN, infinite, huge, tiny and signed-zero coordinates: codes,
    order, splits and bounds are those of the build in separate launches (as a world
    that times its stages makes it) and of the oracle."""
    rng = np.random.default_rng(n + len(kind))
    data = _elements(kind, n, rng)
    flat = data.reshape(-1)
    for v in (np.nan, np.inf, -np.inf, 1e300, -1e300, 5e-324, -0.0):
        flat[rng.integers(0, flat.size, 1 + n // 100)] = v
    kd, ce = O.elements_sphere(data) if kind == "sphere" else O.elements_poly(data)
    for bits, od in ((63, 16), (30, 64)):
        got = []
        for timing in (False, True):
            with CollisionWorld(od, morton_bits=bits, timing=timing) as w:
                o = w.create_collision_object()
                if kind == "sphere":
                    o.set_entity_data_sphere(to_cuda(data))
                else:
                    o.set_entity_data_poly(to_cuda(data))
                o.init_broadphase()
                got.append([*o.sorted(), o.splits(), *o.bounds()])
        ref = O.Object(kd, ce, od=od, morton_bits=bits)
        for x, y in zip(*got):
            assert np.array_equal(x, y, equal_nan=x.dtype == np.float64)
        assert np.array_equal(got[0][0], ref.codes) and np.array_equal(got[0][1], ref.perm)
        assert np.array_equal(got[0][2], ref.splits.astype(np.uint64))
