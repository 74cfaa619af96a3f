"""GPU: sorts at the edges of the radix passes' tiles and of the local sort's range,
every element width, bit-exact and stable vs numpy's stable sort (integer keys)
and the oracle (floats)."""
import numpy as np
import pytest

import massively_amd as m
import oracle
from massively_amd import random as mr

pytestmark = pytest.mark.gpu

EDGES = [1, 1024, 1025, 4096, 4097, 5120, 5121, 8191, 8192, 8193, 10239, 10240, 10241, 3 * 8192 + 5,
         (1 << 18) + 1, 41 * 10240 - 1]


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


@pytest.mark.parametrize("dtype,value", [(np.uint32, np.uint32), (np.uint64, np.uint32), (np.uint64, np.uint64),
                                         (np.uint32, None)])
@pytest.mark.parametrize("spread", ["uniform", "top constant", "one digit full", "two digits"])
def test_sort_local_range(exec_, dtype, value, spread):
    """One pass and local sorts, and inputs whose highest varying digit rules them out."""
    rng = np.random.default_rng(23)
    bits = 8 * np.dtype(dtype).itemsize
    for n in (9000, 100_003, 900_001, 1_500_000):
        k = rng.integers(0, 2**bits, n, dtype=np.uint64)
        if spread == "top constant":
            k &= np.uint64(2 ** (bits - 8) - 1)
        elif spread == "one digit full":  # a run too long for a block
            k[rng.random(n) < 0.5] &= np.uint64(2 ** (bits - 8) - 1)
        elif spread == "two digits":
            k &= np.uint64(0xFF | 0xFF << (bits - 8))
        k = k.astype(dtype)
        order = np.argsort(k, kind="stable")
        dk = exec_.to_device(k)
        if value is None:
            assert np.array_equal(exec_.to_host(m.vector.sort(exec_, dk, m.op.Less)), k[order]), n
            assert np.array_equal(exec_.to_host(m.vector.sort(exec_, dk, m.op.Greater)), k[order][::-1]), n
            continue
        v, s = m.vector.radix_sort_by_key(exec_, dk, exec_.to_device(np.arange(n, dtype=value)), return_keys=True)
        assert np.array_equal(exec_.to_host(v), order.astype(value)), n
        assert np.array_equal(exec_.to_host(s), k[order]), n


@pytest.mark.parametrize("dtype,value", [(np.uint32, np.uint32), (np.uint64, np.uint32), (np.uint64, np.uint64),
                                         (np.uint64, None)])
@pytest.mark.parametrize("values", [(0, 1), (0, 255), (3, 4, 7, 99)])
def test_sort_few_values_in_high_digits(exec_, dtype, value, values):
    """Short sorts whose highest varying digits tell few elements apart: those that
    vary in few bits take more digits at once, those of 0 and 255 leave runs that
    are too long to repair and start over."""
    rng = np.random.default_rng(len(values))
    width = np.dtype(dtype).itemsize
    for n, top in ((17, False), (1500, False), (4096, False), (100_003, True), (300_000, True), (12_000, False)):
        k = rng.integers(0, 256, (n, width), dtype=np.uint8)  # little endian digits
        few = np.array(values, np.uint8)
        for d in range(width - 3 - top, width - top):
            k[:, d] = few[rng.integers(0, few.size, n)]
        k = k.view(dtype).reshape(-1)
        order = np.argsort(k, kind="stable")
        dk = exec_.to_device(k)
        if value is None:
            assert np.array_equal(exec_.to_host(m.vector.sort(exec_, dk, m.op.Less)), k[order]), n
            continue
        v, s = m.vector.radix_sort_by_key(exec_, dk, exec_.to_device(np.arange(n, dtype=value)), return_keys=True)
        assert np.array_equal(exec_.to_host(v), order.astype(value)), n
        assert np.array_equal(exec_.to_host(s), k[order]), n


@pytest.mark.parametrize("dtype,value", [(np.uint64, np.uint32), (np.int64, None), (np.float64, np.uint64)])
@pytest.mark.parametrize("spread", ["uniform", "sorted", "pairs", "runs", "half", "one digit", "many runs",
                                    "few values", "six digits", "seven digits"])
def test_sort_high_digits_and_repair(exec_, dtype, value, spread):
    """Long sorts of 8-byte keys: nothing, pairs, runs of some hundred elements and a
    run of half the keys that differ only in digits the first passes could leave
    out; many runs of 34 beside each other, which the repair gives up on, so that
    the passes start over; digits of ten values each; and seven digits or all of
    them before the keys differ."""
    n = (1 << 23) + 4099
    rng = np.random.default_rng(41)
    few = rng.random(n) < (1e-4 if spread == "runs" else 1e-5)
    low = rng.integers(0, 1 << 16, n, dtype=np.uint64)
    if spread == "pairs":  # one pair of keys in three shares all but 16 bits
        k = rng.permutation(rng.integers(0, 2**46, n, dtype=np.uint64).repeat(2)[:n]) << np.uint64(16)
        k |= np.where(rng.random(n) < 1 / 3, low, np.uint64(0))
    elif spread == "runs":
        k = rng.choice(rng.integers(0, 2**46, 1 << 14, dtype=np.uint64), n) << np.uint64(16)
        k |= np.where(few, low, np.uint64(0))
    elif spread == "half":
        k = rng.integers(0, 2**62, n, dtype=np.uint64)
        hot = rng.random(n) < 0.5
        k[hot] = np.uint64(5 << 40) | np.where(few, low, np.uint64(7))[hot]
    elif spread == "many runs":
        k = rng.integers(0, 2**62, n, dtype=np.uint64)
        runs = (np.uint64(1 << 29) + np.arange(150, dtype=np.uint64).repeat(34)) << np.uint64(32)
        k[rng.choice(n, runs.size, replace=False)] = runs | rng.integers(0, 2**32, runs.size, dtype=np.uint64)
    elif spread == "few values":
        k = rng.integers(0, 10, (n, 8), dtype=np.uint8).view(np.uint64).reshape(-1)
    elif spread == "six digits":  # groups of 512 keys that differ in the lowest two
        k = rng.choice(rng.integers(0, 2**46, n >> 9, dtype=np.uint64), n) << np.uint64(16) | low
    elif spread == "seven digits":  # groups of 16
        k = rng.choice(rng.integers(0, 2**46, n >> 4, dtype=np.uint64), n) << np.uint64(16) | low
    elif spread == "one digit":
        k = rng.integers(0, 256, n, dtype=np.uint64) << np.uint64(48)
    else:
        k = rng.integers(0, 2**62, n, dtype=np.uint64)
    if dtype == np.float64:
        k = (k + np.uint64(1 << 52)).view(np.float64)  # positive normal numbers: ordered as their bits
    else:
        k = k.astype(dtype)
    if spread == "sorted":
        k.sort()
    order = np.argsort(k, kind="stable")
    dk = exec_.to_device(k)
    if value is None:
        assert np.array_equal(exec_.to_host(m.vector.sort(exec_, dk, m.op.Less)), k[order])
        assert np.array_equal(exec_.to_host(m.vector.sort(exec_, dk, m.op.Greater)), k[order][::-1])
        return
    v, s = m.vector.radix_sort_by_key(exec_, dk, exec_.to_device(np.arange(n, dtype=value)), return_keys=True)
    assert np.array_equal(exec_.to_host(v), order.astype(value))
    assert np.array_equal(exec_.to_host(s), k[order])


def test_sort_most_keys_repair_at_the_end():
    """2^32 - 1 keys of 8 bytes, the last 2000 of which differ in the lowest digits
    only: the run to repair ends beside the largest 32-bit index."""
    ex = m.Executor(0)  # its 140 GB go back with it
    n, many = (1 << 32) - 1, 2000
    rng = np.random.default_rng(5)
    last = np.sort(np.uint64(0xFFFFFFFFFF000000) | rng.integers(0, 1 << 24, many, dtype=np.uint64))
    keys = ex.alloc(np.uint64, n)
    for lo in range(0, n, 1 << 31):
        hi = min(n, lo + (1 << 31))
        mr.uniform_u64(ex, 0, 2**63 - 1, lo + 1, keys.slice(lo, hi))
    places = rng.choice(n, many, replace=False).astype(np.uint32)
    m.vector.scatter(ex, ex.to_device(last[::-1].copy()), ex.to_device(np.sort(places)), keys)
    out = m.vector.sort(ex, keys, m.op.Less)
    assert np.array_equal(ex.to_host(out.slice(n - many, n)), last)
    for lo in (0, n // 3, n - (1 << 20)):
        part = ex.to_host(out.slice(lo, lo + (1 << 20)))
        assert np.all(part[:-1] <= part[1:])
    ex.close()
