"""GPU: sorts at the edges of the radix passes' tiles, every element width, bit-exact
and stable vs numpy's stable sort (integer keys) and the oracle (floats)."""
import numpy as np
import pytest

import massively_amd as m
import oracle

pytestmark = pytest.mark.gpu

EDGES = [8191, 8192, 8193, 10239, 10240, 10241, 3 * 8192 + 5, 41 * 10240 - 1]


def _keys(dtype, n, rng, few):
    dtype = np.dtype(dtype)
    if dtype.kind == "f":
        return rng.standard_normal(n).astype(dtype)
    if few:  # many ties: stability shows
        return (rng.integers(0, 37, n).astype(np.uint64) * np.uint64(0x0101010101010101)).astype(dtype)
    return rng.integers(0, 2**64, n, dtype=np.uint64).astype(dtype)


@pytest.mark.parametrize("dtype", [np.uint32, np.int32, np.float32, np.uint64, np.int64])
@pytest.mark.parametrize("value", [None, np.uint32, np.uint64])
def test_sort_tile_edges(exec_, dtype, value):
    rng = np.random.default_rng(17)
    for n in EDGES:
        for few in (False, True):
            k = _keys(dtype, n, rng, few)
            order = (np.argsort(k, kind="stable") if np.dtype(dtype).kind != "f"
                     else oracle.radix_sort_by_key(k, np.arange(n, dtype=np.uint32))[1])
            dk = exec_.to_device(k)
            if value is None:
                assert np.array_equal(exec_.to_host(m.vector.sort(exec_, dk, m.op.Less)), k[order]), n
                continue
            v, s = m.vector.radix_sort_by_key(exec_, dk, exec_.to_device(np.arange(n, dtype=value)), return_keys=True)
            assert np.array_equal(exec_.to_host(v), order.astype(value)), (n, few)
            assert np.array_equal(exec_.to_host(s), k[order]), (n, few)
