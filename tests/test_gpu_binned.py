"""GPU: the binned forms of scatter and gather (large tables), bit-exact vs
numpy indexing: ragged lengths, unaligned slices, tiles that go the direct way
beside binned ones, chunks that overflow, dropped and out-of-range indices."""
import numpy as np
import pytest

import massively_amd as m
from massively_amd import random as mr

pytestmark = pytest.mark.gpu

N = 1 << 23  # the smallest binned scatter


def _order(kind, n, size, rng):
    """n distinct indices below size in the given order."""
    if kind == "random":
        return rng.permutation(size)[:n].astype(np.uint32)
    if kind == "half":  # twice the mean in half of the windows
        return rng.permutation(size // 2)[:n].astype(np.uint32)
    if kind in ("third", "sixth"):  # four chunks of a group; more than the mean that tiles are binned with
        return rng.permutation(size // (3 if kind == "third" else 6))[:n].astype(np.uint32)
    if kind == "streams":  # the places of a stable partition into 256 parts: long rows of one leaf
        part = rng.integers(0, 256, n).astype(np.uint8)
        idx = np.empty(n, np.uint32)
        idx[np.argsort(part, kind="stable")] = np.arange(n, dtype=np.uint32) + (size - n)
        return idx
    if kind.startswith("rows"):  # of some elements: written directly, or not
        w = int(kind[4:])
        return (rng.permutation(size // w)[:n // w + 1, None].astype(np.uint32) * np.uint32(w)
                + np.arange(w, dtype=np.uint32)).reshape(-1)[:n]
    if kind == "reversed":
        return np.arange(size - 1, size - 1 - n, -1, dtype=np.uint32)
    idx = rng.permutation(size)[:n].astype(np.uint32)  # "mixed": sorted and random stretches
    for lo in range(0, n, 100_000):
        if (lo // 100_000) % 2:
            idx[lo:lo + 100_000] = np.sort(idx[lo:lo + 100_000])
    return idx


@pytest.mark.parametrize("dtype,kind,n,size,offset", [
    (np.uint32, "random", N, N, 0),
    (np.uint32, "random", N + 12345, 2 * N + 7, 1),
    (np.uint32, "half", N, 2 * N + 4, 0),
    (np.uint32, "mixed", N + 1, N + 16385, 3),
    (np.uint32, "reversed", N + 16383, 3 * N, 0),
    (np.uint32, "random", 4 * N - 1, 4 * N, 0),
    (np.uint64, "random", N + 4095, N + 8193, 0),
    (np.uint64, "half", N, 2 * N, 1),
    (np.uint64, "mixed", 2 * N + 3, 2 * N + 5, 0),
    (np.uint32, "third", N + 5, 3 * N + 1000, 0),
    (np.uint32, "sixth", N, 6 * N + 9, 1),
    (np.uint64, "third", N, 3 * N + 77, 0),
    (np.uint32, "streams", 4 * N + 3, 4 * N + 3, 0),
    (np.uint64, "streams", N + 1, N + 5, 1),
    (np.uint32, "rows16", N + 7, 2 * N, 1),
    (np.uint32, "rows4", N, 2 * N, 0),
    (np.uint64, "rows8", N + 9, 2 * N, 0),
])
def test_binned_scatter(exec_, dtype, kind, n, size, offset):
    rng = np.random.default_rng(n + size)
    idx = _order(kind, n, size, rng)
    idx[rng.integers(0, n, 1000)] = size + rng.integers(0, 2**20, 1000).astype(np.uint32)  # dropped
    v = rng.integers(0, 2**32, n).astype(dtype)
    before = rng.integers(0, 2**32, size).astype(dtype)
    pad = np.zeros(offset, dtype)
    di = exec_.to_device(np.concatenate([pad.astype(np.uint32), idx])).slice(offset, offset + n)
    dv = exec_.to_device(np.concatenate([pad, v])).slice(offset, offset + n)
    whole = exec_.to_device(np.concatenate([pad, before, pad]))
    m.vector.scatter(exec_, dv, di, whole.slice(offset, offset + size))
    kept = idx < size
    before[idx[kept]] = v[kept]
    assert np.array_equal(exec_.to_host(whole), np.concatenate([pad, before, pad]))


def test_binned_scatter_duplicates(exec_):
    """One of the values aimed at a place ends up there."""
    rng = np.random.default_rng(3)
    idx = rng.integers(0, N, N).astype(np.uint32)
    out = exec_.to_device(np.full(N, 0xFFFFFFFF, np.uint32))
    m.vector.scatter(exec_, exec_.to_device(np.arange(N, dtype=np.uint32)), exec_.to_device(idx), out)
    got = exec_.to_host(out)
    hit = np.zeros(N, bool)
    hit[idx] = True
    assert np.array_equal(got != 0xFFFFFFFF, hit)
    assert np.array_equal(idx[got[hit]], np.flatnonzero(hit))


@pytest.mark.parametrize("dtype", [np.uint32, np.uint64])
@pytest.mark.parametrize("hot", [0.07, 0.9])
def test_binned_scatter_hot_indices(exec_, dtype, hot):
    """Some indices are there many times: one of their values ends up there."""
    n, size = N + 20_000, 3 * N
    rng = np.random.default_rng(int(hot * 100))
    idx = rng.integers(0, size, n).astype(np.uint32)
    few = np.array([0, 5, size - 1], np.uint32)
    idx[rng.random(n) < hot] = few[2]
    idx[rng.random(n) < hot / 4] = few[0]
    out = exec_.to_device(np.full(size, 2**32 - 1, dtype))
    m.vector.scatter(exec_, exec_.to_device(np.arange(n, dtype=dtype)), exec_.to_device(idx), out)
    got = exec_.to_host(out)
    hit = np.zeros(size, bool)
    hit[idx] = True
    assert np.array_equal(got != 2**32 - 1, hit)
    assert np.array_equal(idx[got[hit].astype(np.int64)], np.flatnonzero(hit))


@pytest.mark.parametrize("dtype", [np.uint32, np.uint64])
@pytest.mark.parametrize("n,apart", [(1, 1), (63, 2), (4096, 1), (70_001, 3), (1_000_003, 64), (N + 4097, 16)])
def test_scatter_sorted_indices(exec_, dtype, n, apart):
    """Indices in order, some elements apart, up and down, from unaligned slices."""
    size = n * apart + 5
    up = np.arange(n, dtype=np.uint32) * np.uint32(apart) + np.uint32(2)
    v = np.arange(1, n + 1, dtype=dtype)
    for idx in (up, up[::-1].copy()):
        di = exec_.to_device(np.concatenate([[9], idx]).astype(np.uint32)).slice(1, n + 1)
        out = exec_.to_device(np.zeros(size, dtype))
        m.vector.scatter(exec_, exec_.to_device(np.concatenate([[0], v]).astype(dtype)).slice(1, n + 1), di, out)
        want = np.zeros(size, dtype)
        want[idx] = v
        assert np.array_equal(exec_.to_host(out), want), n


def test_binned_scatter_replays(exec_):
    rng = np.random.default_rng(5)
    v = exec_.to_device(np.arange(N, dtype=np.uint32))
    idx, out = exec_.to_device(rng.permutation(N).astype(np.uint32)), exec_.alloc(np.uint32, N)
    with exec_.capture() as cap:
        m.vector.scatter(exec_, v, idx, out)
    for _ in range(3):
        p = rng.permutation(N).astype(np.uint32)
        m.vector.scatter(exec_, exec_.to_device(p), v, idx)  # idx <- p (v is the identity)
        m.vector.scatter(exec_, exec_.to_device(np.zeros(N, np.uint32)), v, out)
        exec_.sync()
        cap.graph.launch()
        exec_.sync()
        got = exec_.to_host(out)
        assert np.array_equal(got[p], np.arange(N, dtype=np.uint32))


def test_binned_scatter_largest_output():
    """An output of 2^32 - 1 elements, whose last leaf ends past 32 bits."""
    ex = m.Executor(0)  # its 24 GB go back with it
    n, size = 1 << 28, (1 << 32) - 1
    idx = np.arange(n, dtype=np.uint32) * np.uint32(2654435761)  # distinct, in no order
    v, out = ex.alloc(np.uint32, n), ex.alloc(np.uint32, size)
    mr.iota_u32(ex, v, 1)
    for lo in range(0, size, 1 << 31):
        mr.uniform_u32(ex, 0, 0, 1, out.slice(lo, min(size, lo + (1 << 31))))
    di = ex.to_device(idx)
    m.vector.scatter(ex, v, di, out)
    got = ex.to_host(m.vector.gather(ex, out, di))
    kept = idx < size
    assert np.array_equal(got[kept], np.arange(1, n + 1, dtype=np.uint32)[kept])
    ex.close()


@pytest.mark.parametrize("kind,offset,outside", [("random", 0, 0), ("mixed", 1, 500), ("rows", 3, 40),
                                                 ("mostly random", 0, 0)])
def test_binned_gather(exec_, kind, offset, outside):
    """Both ways the looks decide, and tiles that go directly in the binned form."""
    n, size = (1 << 27) + 40_000, (1 << 27) - 7
    rng = np.random.default_rng(offset)
    idx = np.empty(n + offset, np.uint32)
    step = 1 << 24
    for lo in range(0, n + offset, step):  # (a permutation of 2^27 costs the test 10 s)
        k = min(step, n + offset - lo)
        idx[lo:lo + k] = rng.integers(0, size, k, dtype=np.uint32)
    if kind == "mixed":
        for lo in range(0, n - 50_000, 1 << 20):
            idx[lo:lo + 50_000] = np.arange(lo % size, lo % size + 50_000) % size
    elif kind == "rows":  # of 64 elements: a direct gather
        rows = idx[:(n + offset) // 64] // np.uint32(64) * np.uint32(64)
        idx[:rows.size * 64].reshape(-1, 64)[:] = rows[:, None] + np.arange(64, dtype=np.uint32)
    elif kind == "mostly random":  # one tile in eight is sorted
        for lo in range(0, n - 65536, 8 * 32768):
            idx[lo:lo + 32768] = np.sort(idx[lo:lo + 32768])
            idx[lo + 32768:lo + 65536] = np.arange(32768, dtype=np.uint32) + np.uint32(lo % (size - 32768))
    idx[rng.integers(0, n, outside)] = size + 3
    v = rng.integers(0, 2**32, size, dtype=np.uint32)
    di = exec_.to_device(idx).slice(offset, offset + n)
    got = exec_.to_host(m.vector.gather(exec_, exec_.to_device(v), di))
    j = idx[offset:]
    inside = j < size
    assert np.array_equal(got, np.where(inside, v[np.where(inside, j, 0)], 0))
