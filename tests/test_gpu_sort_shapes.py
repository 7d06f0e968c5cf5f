"""The radix sort at the sizes where its shapes and tiles end, on random keys,
keys of few distinct values (ties keep their order) and keys that differ in one
digit, against numpy's stable sort."""
import numpy as np
import pytest

from distbvh_amd import CollisionWorld
from helpers import from_cuda, to_cuda

pytestmark = pytest.mark.gpu

WIDE = 3 << 19  # the first size of the wide pass shape
SIZES = [1, 2, 63, 64, 65, 255, 1023, 1024, 1025, 2047, 2049, 4095, 4096, 4097, 8191, 8192, 8193, 12289, 40961,
         WIDE - 1, WIDE, WIDE + 8191, WIDE + 8193]


@pytest.fixture(scope="module")
def world():
    import torch
    assert torch.cuda.is_available(), "GPU test needs a GPU"
    with CollisionWorld(1) as w:
        yield w


def _keys(kind, n, dtype, rng):
    bits = 8 * np.dtype(dtype).itemsize
    if kind == "random":
        return rng.integers(0, 2 ** bits, n, dtype=dtype, endpoint=False)
    if kind == "few":
        return rng.integers(0, 5, n).astype(dtype) * dtype(0x01010101)
    if kind == "one_digit":
        return (rng.integers(0, 256, n).astype(dtype) << dtype(8)) | dtype(0x42)
    return np.full(n, 7, dtype)  # equal


@pytest.mark.parametrize("payload", [True, False])
@pytest.mark.parametrize("dtype", [np.uint64, np.uint32])
@pytest.mark.parametrize("n", SIZES)
def test_sort_at_shape_edges(world, n, dtype, payload):
    rng = np.random.default_rng(n)
    for kind in ("random", "few", "one_digit", "equal"):
        keys = _keys(kind, n, dtype, rng)
        vals = rng.integers(0, 2 ** 32, n, dtype=np.uint32)
        order = np.argsort(keys, kind="stable")
        tk, tv = to_cuda(keys), (to_cuda(vals) if payload else None)
        world.sort(tk, tv)
        assert np.array_equal(from_cuda(tk, dtype), keys[order]), kind
        if payload:
            assert np.array_equal(from_cuda(tv, np.uint32), vals[order]), kind
