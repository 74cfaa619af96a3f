"""GPU: library calls captured into a HIP graph and replayed.

Each replay runs after eager work that rewrites the inputs (the library's
generator), and every replay's outputs are checked against the oracle, so a
replay that reused stale lookback state or scratch would fail.
"""
import numpy as np
import pytest

import massively_amd as m
import oracle
from massively_amd import random as mr
from massively_amd import seg, serve

pytestmark = pytest.mark.gpu


def test_graph_replays_scan_seg_sort_and_jobs(exec_):
    ex = exec_
    n = 300000
    x = ex.alloc(np.uint32, n)
    lengths = np.random.default_rng(5).integers(0, 3000, 200)
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)
    ns = int(off[-1])
    sg = seg.Segmentation.from_offsets(ex, ex.to_device(off))
    k = ex.alloc(np.uint32, ns)
    v = ex.alloc(np.uint32, ns)
    mr.iota_u32(ex, v)
    small = ex.alloc(np.uint32, 5000)
    small_out = ex.alloc(np.uint32, 5000)
    skeys = ex.alloc(np.uint32, 3000)
    skeys_out = ex.alloc(np.uint32, 3000)
    jobs = [serve.Job("exclusive_scan", small, small_out, op=m.op.Add, init=7),
            serve.Job("sort_by_key", skeys, None, op=m.op.Less, out2=skeys_out)]
    ex.sync()
    with ex.capture() as cap:
        y = m.vector.inclusive_scan(ex, x, m.op.Add)
        srt = seg.ForEachSegment(seg.Sort(m.op.Less)).run(ex, seg.SegmentIterator((k, v), sg))
        serve.run_jobs(ex, jobs)
    g = cap.graph
    with pytest.raises(m.Error):
        with ex.capture():
            ex.to_host(x)
    for rep in range(4):
        mr.uniform_u32(ex, 0, 1000, 40 + rep, x)
        mr.uniform_u32(ex, 0, 50, 60 + rep, k)
        mr.uniform_u32(ex, 0, 2**32 - 1, 80 + rep, small)
        mr.uniform_u32(ex, 0, 99, 90 + rep, skeys)
        ex.sync()
        g.launch()
        ex.sync()
        hx = oracle.uniform_u32(0, 1000, 40 + rep, n)
        assert ex.to_host(y).tobytes() == oracle.inclusive_scan(hx, "add").tobytes(), rep
        hk = oracle.uniform_u32(0, 50, 60 + rep, ns)
        perm = oracle.seg_sort_perm(hk, off, "less")
        assert ex.to_host(srt.values[0]).tobytes() == hk[perm].tobytes(), rep
        assert ex.to_host(srt.values[1]).tobytes() == perm.astype(np.uint32).tobytes(), rep
        hs = oracle.uniform_u32(0, 2**32 - 1, 80 + rep, 5000)
        assert ex.to_host(small_out).tobytes() == oracle.exclusive_scan(hs, 7, "add").tobytes(), rep
        hk2 = oracle.uniform_u32(0, 99, 90 + rep, 3000)
        assert ex.to_host(skeys_out).tobytes() == np.sort(hk2, kind="stable").tobytes(), rep
    g.close()


def test_graph_replays_long_sort_of_wide_keys(exec_):
    """The digits that get a pass are chosen on every replay (starting over: below)."""
    n = (1 << 21) + 77
    k, v = exec_.alloc(np.uint64, n), exec_.to_device(np.arange(n, dtype=np.uint32))
    mr.uniform_u64(exec_, 0, 9, 1, k)
    exec_.sync()
    with exec_.capture() as cap:
        out, srt = m.vector.radix_sort_by_key(exec_, k, v, return_keys=True)
    rng = np.random.default_rng(3)
    uniform = rng.integers(0, 2**63, n, dtype=np.uint64)
    half = uniform.copy()  # one key in half of the places, a few of them off in the lowest bits
    half[rng.random(n) < 0.5] = 5 << 40
    half[half == 5 << 40] += (rng.random(int((half == 5 << 40).sum())) < 1e-5).astype(np.uint64)
    for rep, h in enumerate((uniform, half, uniform & np.uint64(1023), uniform[::-1].copy(), half)):
        m.vector.scatter(exec_, exec_.to_device(h), v, k)
        exec_.sync()
        cap.graph.launch()
        exec_.sync()
        order = np.argsort(h, kind="stable")
        assert np.array_equal(exec_.to_host(out), order.astype(np.uint32)), rep
        assert np.array_equal(exec_.to_host(srt), h[order]), rep
    cap.graph.close()


def test_graph_replays_sort_that_starts_over(exec_):
    """Between replays that need no repair, one whose repair gives up (many runs of 34
    keys beside each other)."""
    n = (1 << 23) + 11
    rng = np.random.default_rng(9)
    plain = rng.integers(0, 2**62, n, dtype=np.uint64)
    runs = (np.uint64(1 << 29) + np.arange(150, dtype=np.uint64).repeat(34)) << np.uint64(32)
    many = plain.copy()
    many[rng.choice(n, runs.size, replace=False)] = runs | rng.integers(0, 2**32, runs.size, dtype=np.uint64)
    k, v = exec_.alloc(np.uint64, n), exec_.to_device(np.arange(n, dtype=np.uint32))
    exec_.sync()
    with exec_.capture() as cap:
        out, srt = m.vector.radix_sort_by_key(exec_, k, v, return_keys=True)
    for rep, h in enumerate((plain, many, plain, many)):
        m.vector.scatter(exec_, exec_.to_device(h), v, k)
        exec_.sync()
        cap.graph.launch()
        exec_.sync()
        order = np.argsort(h, kind="stable")
        assert np.array_equal(exec_.to_host(out), order.astype(np.uint32)), rep
        assert np.array_equal(exec_.to_host(srt), h[order]), rep
    cap.graph.close()


@pytest.mark.parametrize("beside", ["scans", "device-wide"])
def test_graph_replays_forked_jobs(exec_, beside):
    """A captured batch whose long sort runs on the second stream, beside scans of
    its table and device-wide jobs."""
    ex, n = exec_, 1 << 14
    k, ok = ex.alloc(np.uint64, n), ex.alloc(np.uint64, n)
    v, ov = ex.to_device(np.arange(n, dtype=np.uint32)), ex.alloc(np.uint32, n)
    sizes = [1 << 17, 70_000, 5000] if beside == "scans" else [1 << 18, 150_000, 200_001, 140_000]
    xs, ys = [ex.alloc(np.uint32, c) for c in sizes], [ex.alloc(np.uint32, c) for c in sizes]
    jobs = [serve.Job("sort_by_key", k, ov, op=m.op.Less, inp2=v, out2=ok)]
    jobs += [serve.Job("inclusive_scan", x, y, op=m.op.Add) for x, y in zip(xs, ys)]
    serve.run_jobs(ex, jobs)  # (tunes its launches outside of the capture)
    ex.sync()
    with ex.capture() as cap:
        serve.run_jobs(ex, jobs)
    for rep in range(4):
        mr.uniform_u64(ex, 0, 1 << 40, 7 + rep, k)
        for x in xs:
            mr.uniform_u32(ex, 0, 1000, 40 + rep, x)
        ex.sync()
        cap.graph.launch()
        ex.sync()
        hk = ex.to_host(k)
        order = np.argsort(hk, kind="stable")
        assert np.array_equal(ex.to_host(ok), hk[order]), rep
        assert np.array_equal(ex.to_host(ov), order.astype(np.uint32)), rep
        for x, y in zip(xs, ys):
            assert np.array_equal(ex.to_host(y), np.cumsum(ex.to_host(x), dtype=np.uint32)), rep
    cap.graph.close()
