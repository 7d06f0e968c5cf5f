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
