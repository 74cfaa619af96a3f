"""The workloads whose speed is measured, as calls of the package's public API.

Each case is one call (or one batch of jobs) of ``massively_amd.vector``,
``massively_amd.seg`` or ``massively_amd.serve`` on device-resident data, over
the sizes, data types and options of the benchmark configurations and of the
tests. Inputs are torch tensors that the library borrows with
``Executor.wrap``; results are returned as torch views of the library's device
vectors. Unsigned columns are held in torch as the signed type of their width.
"""
import random

import numpy as np
import torch

import massively_amd as m
from massively_amd import seg, serve

NP = {"u32": np.uint32, "i32": np.int32, "f32": np.float32, "u64": np.uint64, "i64": np.int64, "f64": np.float64}
TORCH = {"u32": torch.int32, "i32": torch.int32, "f32": torch.float32,
         "u64": torch.int64, "i64": torch.int64, "f64": torch.float64}
SIZE = {"u32": 4, "i32": 4, "f32": 4, "u64": 8, "i64": 8, "f64": 8}
TYPESTR = {4: {"u": "<i4", "i": "<i4", "f": "<f4"}, 8: {"u": "<i8", "i": "<i8", "f": "<f8"}}
OPS = {"add": m.op.Add, "min": m.op.Min, "max": m.op.Max, "xor": m.op.Xor}

_executor = None


def executor():
    """The program's one executor (a stream and an allocator)."""
    global _executor
    if _executor is None:
        _executor = m.Executor(0)
    return _executor


class _Borrowed:
    """A device vector's memory for torch; keeps the vector alive."""

    def __init__(self, vec, n):
        dt = vec.dtype
        self.vec = vec
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": TYPESTR[dt.itemsize][dt.kind],
                                         "data": (vec.device_ptr, False), "strides": None, "version": 3}


def tensor(vec):
    """A device vector as a torch tensor of its length (a length that only the
    device knows, as after a selection, is read back)."""
    n = vec.len()
    if n == 0:
        return torch.empty(0, dtype=TORCH["u32"], device="cuda")
    return torch.as_tensor(_Borrowed(vec, n), device="cuda")


# ---------------------------------------------------------------- cases


def listed():
    return [
        # A sum of a few thousand values whose scalar the program waits for.
        {"name": "reduce_small", "kind": "reduce", "dtype": "f32", "op": "add", "n": 5000, "offset": 0},
        # A prefix sum of 10 million floats, the size of the reference's own table.
        {"name": "scan_f32_10m", "kind": "scan", "dtype": "f32", "op": "add", "n": 10_000_000, "exclusive": False,
         "offset": 0},
        # The scan configuration: 2^28 u32, add.
        {"name": "scan_u32_2^28", "kind": "scan", "dtype": "u32", "op": "add", "n": 1 << 28, "exclusive": False,
         "offset": 0},
        # The plain sort configuration: a permutation that sorts 2^20 u32 keys.
        {"name": "sort_u32_2^20", "kind": "sort", "dtype": "u32", "value": "u32", "n": 1 << 20, "spread": "uniform",
         "keys": False},
        # The headline sort: 2^28 u32 keys with a u32 payload.
        {"name": "sort_u32_2^28", "kind": "sort", "dtype": "u32", "value": "u32", "n": 1 << 28, "spread": "uniform",
         "keys": False},
        # 2^27 u64 keys with few distinct, skewed values and a u32 payload.
        {"name": "sort_u64_2^27", "kind": "sort", "dtype": "u64", "value": "u32", "n": 1 << 27, "spread": "zipf",
         "keys": False},
        # Filtering a column by a flag column, half of it kept.
        {"name": "copy_where_2^28", "kind": "select", "dtype": "u32", "form": "stencil", "keep": 0.5, "n": 1 << 28,
         "offset": 0},
        # The intersection of two sorted sets that share a quarter.
        {"name": "intersect_2x2^27", "kind": "ordered", "op": "intersection", "dtype": "u32", "n": 1 << 27,
         "m": 1 << 27, "overlap": 0.25, "repeat": 0},
        # Reading and writing a column in the order of a random permutation.
        {"name": "gather_2^28", "kind": "gather", "dtype": "u32", "n": 1 << 28, "table": 1 << 28, "order": "random"},
        {"name": "scatter_2^28", "kind": "scatter", "dtype": "u32", "n": 1 << 28, "table": 1 << 28, "order": "random"},
        # Sorting every one of a million ragged rows by key.
        {"name": "seg_sort_2^26", "kind": "seg", "op": "sort", "dtype": "u32", "value": "f32", "n": 1 << 26,
         "segments": 1 << 20},
        # One batch of independent small jobs of every family, as a server collects them.
        {"name": "jobs_96", "kind": "jobs", "jobs": 96, "low": 10, "high": 17, "mix": 1},
    ]


def _size(rng, low, high):
    """A length between 2^low and 2^high, spread over the logarithm, mostly odd or ragged."""
    n = int(2.0 ** rng.uniform(low, high))
    return n if rng.random() < 0.8 else max(1 << low, n & ~1023)


def draw(rng):
    kind = rng.choice(["reduce", "scan", "sort", "select", "ordered", "gather", "scatter", "seg", "jobs"])
    offset = rng.choice([0, 0, 0, 1])
    if kind in ("reduce", "scan"):
        dtype = rng.choice(["u32", "f32", "u64", "f64", "i32"])
        n = _size(rng, 10, 28 if SIZE[dtype] == 4 else 27)
        c = {"kind": kind, "dtype": dtype, "op": rng.choice(["add", "add", "max"]), "n": n, "offset": offset}
        return c if kind == "reduce" else {**c, "exclusive": rng.random() < 0.5}
    if kind == "sort":
        dtype = rng.choice(["u32", "u64", "f32", "i32", "i64"])
        value = rng.choice(["u32", "u32", "u64", "none"])
        top = (28 if SIZE[dtype] == 4 else 27) - (1 if value == "u64" else 0)
        spread = rng.choice(["uniform", "uniform", "zipf", "narrow"] if dtype != "f32" else ["uniform"])
        return {"kind": kind, "dtype": dtype, "value": value, "n": _size(rng, 10, top), "spread": spread,
                "keys": value != "none" and rng.random() < 0.3}
    if kind == "select":
        dtype = rng.choice(["u32", "f32", "u64"])
        return {"kind": kind, "dtype": dtype, "form": rng.choice(["stencil", "predicate"]),
                "keep": round(rng.uniform(0.01, 0.99), 3), "n": _size(rng, 10, 28 if SIZE[dtype] == 4 else 27),
                "offset": offset}
    if kind == "ordered":
        dtype = rng.choice(["u32", "u64"])
        n = _size(rng, 10, 27 if dtype == "u32" else 26)
        return {"kind": kind, "op": rng.choice(["merge", "intersection", "difference", "union"]), "dtype": dtype,
                "n": n, "m": max(1, int(n * rng.uniform(0.25, 1.0))), "overlap": round(rng.uniform(0.05, 0.9), 3),
                "repeat": rng.choice([0, 4, 32])}
    if kind in ("gather", "scatter"):
        dtype = rng.choice(["u32", "f32", "u64"])
        table = _size(rng, 10, 28 if SIZE[dtype] == 4 else 27)
        return {"kind": kind, "dtype": dtype, "table": table, "n": max(1, int(table * rng.uniform(0.25, 1.0))),
                "order": rng.choice(["random", "random", "reverse"])}
    if kind == "seg":
        n = _size(rng, 12, 26)
        op = rng.choice(["scan", "reduce", "sort"])
        dtype = rng.choice(["u32", "f32", "u64"])
        return {"kind": kind, "op": op, "dtype": dtype, "value": rng.choice(["f32", "none"]) if op == "sort" else "none",
                "n": n, "segments": max(1, n // int(2.0 ** rng.uniform(3, 10)))}
    return {"kind": "jobs", "jobs": rng.randint(8, 128), "low": 10, "high": rng.randint(12, 17), "mix": rng.randint(2, 1 << 20)}


# ---------------------------------------------------------------- inputs


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bits(dtype, n, g):
    """Uniform bits for whole numbers, standard normal values for floats (keys and payloads)."""
    if dtype in ("f32", "f64"):
        return torch.randn(n, dtype=TORCH[dtype], device="cuda", generator=g)
    lim = 1 << (8 * SIZE[dtype] - 1)
    return torch.randint(-lim, lim - 1, (n,), dtype=TORCH[dtype], device="cuda", generator=g)


def _addends(dtype, n, g):
    """Values a program sums: counts below 1024, weights in [0, 1)."""
    if dtype in ("f32", "f64"):
        return torch.rand(n, dtype=TORCH[dtype], device="cuda", generator=g)
    return torch.randint(0, 1024, (n,), dtype=TORCH[dtype], device="cuda", generator=g)


def _keys(case, g):
    n, dtype = case["n"], case["dtype"]
    if case["spread"] == "uniform":
        return _bits(dtype, n, g)
    if case["spread"] == "narrow":  # the top byte is the same everywhere
        return torch.bitwise_and(_bits(dtype, n, g), (1 << (8 * SIZE[dtype] - 8)) - 1)
    # Zipf s = 1.1 over 2^20 values spread over the key range.
    cdf = torch.arange(1, (1 << 20) + 1, dtype=torch.float64, device="cuda").pow(-1.1).cumsum(0)
    cdf /= cdf[-1].clone()
    out = torch.empty(n, dtype=torch.int64, device="cuda")
    for lo in range(0, n, 1 << 26):
        hi = min(n, lo + (1 << 26))
        out[lo:hi] = torch.searchsorted(cdf, torch.rand(hi - lo, dtype=torch.float64, device="cuda", generator=g))
    out = out * -7046029254386353131  # an odd multiplier: distinct ranks give distinct keys
    return out if SIZE[dtype] == 8 else (out >> 32).to(torch.int32)


def _distinct(dtype, n, g):
    """n distinct values in no order: a bijective mix of consecutive numbers."""
    bits = 8 * SIZE[dtype]
    mask, first = (1 << bits) - 1 if bits == 32 else -1, int(torch.randint(0, 1 << 31, (1,), device="cuda", generator=g))
    x = (torch.arange(n, dtype=torch.int64, device="cuda") + first) & mask
    for mul in (0x7FEB352D, 0x846CA68B):
        x = x ^ ((x >> (bits // 2)) & ((1 << (bits // 2)) - 1))
        x = (x * (mul if bits == 32 else mul * 0x9E3779B9 | 1)) & mask
    x = x ^ ((x >> (bits // 2)) & ((1 << (bits // 2)) - 1))
    return x.to(TORCH[dtype])


def _chosen(n, keep, g):
    """A random choice of a `keep` share of n places."""
    return torch.randperm(n, device="cuda", generator=g) < int(keep * n)


def _wrap(t, dtype):
    return executor().wrap(t.data_ptr(), NP[dtype], t.numel())


def _sorted_unsigned(t):
    """Sorted by the unsigned value of the bits."""
    low = torch.iinfo(t.dtype).min
    return torch.sort(t ^ low).values ^ low


def _offsets(case, g):
    """Row starts of ragged rows: log-normal lengths, 2% of them empty."""
    s, n = case["segments"], case["n"]
    w = torch.exp(1.1774 * torch.randn(s, dtype=torch.float64, device="cuda", generator=g)).clamp_(max=2048.0)
    w[torch.rand(s, device="cuda", generator=g) < 0.02] = 0.0
    w[-1] += 0.5
    ends = torch.cumsum(w, 0)
    ends = torch.floor(ends * (n / ends[-1])).to(torch.int64).clamp_(max=n)
    ends[-1] = n
    return torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), ends]).to(torch.int32)


def _job_list(case):
    """(kind, dtype, n, place) of a batch's jobs, and the length of the buffers
    they are slices of; jobs start at multiples of 64 elements."""
    rng = random.Random(case["mix"])
    jobs, used = [], {}
    for _ in range(case["jobs"]):
        kind = rng.choice(["inclusive_scan", "reduce", "copy_where", "sort_by_key"])
        dtype = rng.choice(["u32", "u64", "f32"])
        n = int(2.0 ** rng.uniform(case["low"], case["high"]))
        place = used.get(dtype, 0)
        used[dtype] = place + (n + 63) // 64 * 64
        jobs.append((kind, dtype, n, place))
    return jobs, used


def _prepare_jobs(case, g):
    jobs, used = _job_list(case)
    ex, span = executor(), max(used.values())
    inp = {d: (_addends if d == "f32" else _bits)(d, k, g) for d, k in used.items()}
    # Scans and sums apart from moved elements, which are never rounded.
    out = {f"{what}_{d}": torch.zeros(k, dtype=TORCH[d], device="cuda") for d, k in used.items()
           for what in ("sums", "moved")}
    # Sorts' payload (a position each), one for each dtype.
    pos = torch.arange(span, dtype=torch.int32, device="cuda")
    pay = {d: torch.zeros(k, dtype=torch.int32, device="cuda") for d, k in used.items()}
    count = torch.zeros(64 * len(jobs), dtype=torch.int32, device="cuda")
    todo = []
    for i, (kind, d, n, at) in enumerate(jobs):
        def piece(t, dtype, k=n, at=at):
            return ex.wrap(t.data_ptr() + at * SIZE[dtype], NP[dtype], k)

        x, dst = piece(inp[d], d), out[("moved_" if kind in ("copy_where", "sort_by_key") else "sums_") + d]
        if kind == "inclusive_scan":
            job = serve.Job(kind, x, piece(dst, d), op=m.op.Add)
        elif kind == "reduce":
            job = serve.Job(kind, x, piece(dst, d, 1), op=m.op.Add, init=0)
        elif kind == "copy_where":
            pred = {"u32": m.op.Lt(1 << 31), "u64": m.op.Lt(1 << 63), "f32": m.op.Lt(0.5)}[d]
            job = serve.Job(kind, x, piece(dst, d), pred=pred, out2=piece(count, "u32", 1, 64 * i))
        else:
            job = serve.Job(kind, x, piece(pay[d], "u32"), inp2=ex.wrap(pos.data_ptr(), NP["u32"], n),
                            out2=piece(dst, d))
        todo.append(job)
    return {"jobs": todo, "out": {**out, **{f"payload_{d}": t for d, t in pay.items()}, "counts": count},
            "hold": (inp, pos)}


def prepare(case, seed):
    g, kind, ex = _generator(seed), case["kind"], executor()
    s = {"case": case}
    if kind in ("reduce", "scan"):
        s["x"] = _addends(case["dtype"], case["n"] + case["offset"], g)
        s["in"] = _wrap(s["x"], case["dtype"]).slice(case["offset"], case["offset"] + case["n"])
    elif kind == "sort":
        s["k"] = _keys(case, g)
        s["keys"] = _wrap(s["k"], case["dtype"])
        if case["value"] != "none":
            s["v"] = torch.arange(case["n"], dtype=TORCH[case["value"]], device="cuda")
            s["values"] = _wrap(s["v"], case["value"])
    elif kind == "select":
        n, off = case["n"], case["offset"]
        kept = torch.cat([torch.zeros(off, dtype=torch.bool, device="cuda"), _chosen(n, case["keep"], g)])
        s["x"] = _bits(case["dtype"], n + off, g)
        if case["form"] == "stencil":
            s["f"] = kept.to(torch.int32)
            s["flags"] = _wrap(s["f"], "u32").slice(off, off + n)
        elif case["dtype"] == "f32":  # kept: below zero
            s["x"], s["pred"] = torch.where(kept, -1.0 - s["x"].abs(), s["x"].abs()), m.op.Lt(0.0)
        else:  # kept: the top bit set
            top = torch.iinfo(s["x"].dtype).min
            s["x"] = torch.where(kept, s["x"] | top, s["x"] & ~top)
            s["pred"] = m.op.Ge(1 << (8 * SIZE[case["dtype"]] - 1))
        s["in"] = _wrap(s["x"], case["dtype"]).slice(off, off + n)
    elif kind == "ordered":
        pool = _distinct(case["dtype"], case["n"] + case["m"], g)
        if case["repeat"]:  # one value in so many is there twice
            pool[case["repeat"]::case["repeat"]] = pool[case["repeat"] - 1:-1:case["repeat"]].clone()
        shared = int(case["overlap"] * case["m"])
        s["a"] = _sorted_unsigned(pool[:case["n"]])
        s["b"] = _sorted_unsigned(pool[case["n"] - shared:case["n"] - shared + case["m"]])
        s["left"], s["right"] = _wrap(s["a"], case["dtype"]), _wrap(s["b"], case["dtype"])
    elif kind in ("gather", "scatter"):
        n, t = case["n"], case["table"]
        i = torch.randperm(t, device="cuda", generator=g) if case["order"] == "random" else torch.arange(t - 1, -1, -1, device="cuda")
        s["i"] = i[:n].to(torch.int32)
        s["index"] = _wrap(s["i"], "u32")
        s["x"] = _bits(case["dtype"], t if kind == "gather" else n, g)
        s["values"] = _wrap(s["x"], case["dtype"])
        if kind == "scatter":
            s["out"] = torch.zeros(t, dtype=TORCH[case["dtype"]], device="cuda")
            s["to"] = _wrap(s["out"], case["dtype"])
    elif kind == "seg":
        s["o"] = _offsets(case, g)
        s["segments"] = seg.Segmentation.from_offsets(ex, _wrap(s["o"], "u32"))
        s["x"] = (_bits if case["op"] == "sort" else _addends)(case["dtype"], case["n"], g)
        s["values"] = _wrap(s["x"], case["dtype"])
        if case["value"] != "none":
            s["p"] = _bits(case["value"], case["n"], g)
            s["values"] = (s["values"], _wrap(s["p"], case["value"]))
    else:
        s.update(_prepare_jobs(case, g))
    torch.cuda.synchronize()  # the inputs are made on torch's stream, the calls run on the executor's
    return s


# ---------------------------------------------------------------- one pass


def run(state):
    ex, case = executor(), state["case"]
    kind = case["kind"]
    if kind == "reduce":
        return m.vector.reduce(ex, state["in"], 0, OPS[case["op"]])
    if kind == "scan":
        if case["exclusive"]:
            return tensor(m.vector.exclusive_scan(ex, state["in"], 0, OPS[case["op"]]))
        return tensor(m.vector.inclusive_scan(ex, state["in"], OPS[case["op"]]))
    if kind == "sort":
        if case["value"] == "none":
            return tensor(m.vector.sort(ex, state["keys"], m.op.Less))
        if case["keys"]:
            v, k = m.vector.radix_sort_by_key(ex, state["keys"], state["values"], return_keys=True)
            return tensor(v), tensor(k)
        return tensor(m.vector.radix_sort_by_key(ex, state["keys"], state["values"]))
    if kind == "select":
        if case["form"] == "stencil":
            return tensor(m.vector.copy_where(ex, state["in"], state["flags"]))
        return tensor(m.vector.copy_where_if(ex, state["in"], state["in"], state["pred"]))
    if kind == "ordered":
        f = m.vector.merge if case["op"] == "merge" else getattr(m.vector, "set_" + case["op"])
        return tensor(f(ex, state["left"], state["right"], m.op.Less))
    if kind == "gather":
        return tensor(m.vector.gather(ex, state["values"], state["index"]))
    if kind == "scatter":
        m.vector.scatter(ex, state["values"], state["index"], state["to"])
        return state["out"]
    if kind == "seg":
        alg = {"scan": seg.InclusiveScan(m.op.Add), "reduce": seg.Reduce(m.op.Add, 0), "sort": seg.Sort(m.op.Less)}[case["op"]]
        r = seg.ForEachSegment(alg).run(ex, seg.SegmentIterator(state["values"], state["segments"]))
        if case["op"] == "reduce":
            return tensor(r)
        return tuple(tensor(v) for v in r.values) if isinstance(r.values, tuple) else tensor(r.values)
    serve.run_jobs(ex, state["jobs"])
    return state["out"]


def work(case):
    kind = case["kind"]
    if kind == "jobs":
        total = 0
        for job, d, n, _ in _job_list(case)[0]:
            w = SIZE[d]
            total += {"inclusive_scan": 2 * w * n, "reduce": w * n, "copy_where": 1.5 * w * n, "sort_by_key": (2 * w + 8) * n}[job]
        return {"bytes": total, "flops": 0}
    n, w = case["n"], SIZE[case["dtype"]]
    if kind == "reduce":
        return {"bytes": w * n, "flops": n}
    if kind == "scan":
        return {"bytes": 2 * w * n, "flops": n}
    if kind == "sort":
        v = 0 if case["value"] == "none" else SIZE[case["value"]]
        return {"bytes": n * (w + 2 * v + (w if case["keys"] or not v else 0)), "flops": 0}
    if kind == "select":
        return {"bytes": n * (w * (1 + case["keep"]) + (4 if case["form"] == "stencil" else 0)), "flops": 0}
    if kind == "ordered":
        shared = int(case["overlap"] * case["m"])
        both = n + case["m"]
        out = {"merge": both, "intersection": shared, "difference": n - shared, "union": both - shared}[case["op"]]
        return {"bytes": w * (both + out), "flops": 0}
    if kind in ("gather", "scatter"):
        return {"bytes": (4 + 2 * w) * n, "flops": 0}
    offsets = 4 * (case["segments"] + 1)
    if case["op"] == "reduce":
        return {"bytes": w * n + offsets + w * case["segments"], "flops": n}
    v = 0 if case["value"] == "none" else SIZE[case["value"]]
    return {"bytes": 2 * (w + v) * n + offsets, "flops": n if case["op"] == "scan" else 0}


# ---------------------------------------------------------------- results


def _sums_floats(case):
    if case["kind"] in ("reduce", "scan"):
        return case["dtype"] if case["op"] == "add" else None
    if case["kind"] == "seg":
        return case["dtype"] if case["op"] != "sort" else None
    return "f32" if case["kind"] == "jobs" else None


def tolerance(case):
    """Float sums may be formed in another order (one order is up to about 2e-7
    off the sum in 64 bits for f32); everything else is moved or wrapped and has
    one right answer."""
    d = _sums_floats(case)
    if d == "f32":
        return {"rel": 1e-6, "max": 1e-5}
    if d == "f64":
        return {"rel": 2e-15, "max": 2e-14}
    return "exact"


def exact(case, seed):
    d = _sums_floats(case)
    if d not in ("f32", "f64"):
        return None
    s = prepare(case, seed)
    if case["kind"] == "jobs":
        sums = torch.zeros(s["out"]["sums_f32"].numel(), dtype=torch.float64, device="cuda") if "sums_f32" in s["out"] else None
        for kind, dt, n, at in _job_list(case)[0]:
            if dt == "f32" and kind in ("inclusive_scan", "reduce"):
                x = s["hold"][0]["f32"][at:at + n].to(torch.float64)
                if kind == "reduce":
                    sums[at] = x.sum()
                else:
                    sums[at:at + n] = x.cumsum(0)
        return {k: (sums if k == "sums_f32" else None) for k in s["out"]}
    x = s["x"].to(torch.float64)
    if case["kind"] == "reduce":
        return float(x[case["offset"]:].sum())
    if case["kind"] == "scan":
        c = x[case["offset"]:].cumsum(0)
        return torch.cat([torch.zeros(1, dtype=c.dtype, device="cuda"), c[:-1]]) if case["exclusive"] else c
    o = s["o"].to(torch.int64)
    before = torch.cat([torch.zeros(1, dtype=x.dtype, device="cuda"), x.cumsum(0)])
    if case["op"] == "reduce":
        return before[o[1:]] - before[o[:-1]]
    row = torch.searchsorted(o[1:].contiguous(), torch.arange(case["n"], device="cuda"), right=True)
    return before[1:] - before[o[:-1][row]]
