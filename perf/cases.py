"""Performance cases: batched interval searches through the package's public entry points.

A case is a dict of plain values; its "kind" names the call:

  search      a batch on device tensors: plan -> offsets -> the total, read back -> fill
  count       the overlap counts of a batch on device tensors
  coverage    count and covered length of a batch (int32 coordinates)
  any         has_overlaps of a batch
  build       an index built from device tensors
  host        a batch of host arrays, CSR result in host memory
  one         queries asked one at a time
  sets        one batch over many resident indexes (a set table)
  intersect   the pieces of a join of two interval sets on device tensors

Position lists go to an output buffer that the program keeps from batch to batch (made
larger when a batch's total asks for it); what lies past the total stays zero.

Intervals and queries follow the package's own generators (workload.cpp), drawn on the GPU:
"lognormal" (starts uniform on [0, 2.5e8), lengths LogNormal(6, 1.5), query lengths
LogNormal(7, 1)) and "hotspots" (70 % uniform on [0, 3e9) and 30 % from 200 Gaussian
hotspots, 20 % of the intervals log-uniform in [1e5, 1e7], 1 % of the queries wide).
"""
import ctypes
import math

import numpy as np
import torch

import superintervals_amd as sia

SPAN = {"lognormal": 250_000_000, "hotspots": 3_000_000_000}
N_SETS = 24


def listed():
    return [
        # a program that asks one query at a time, as the reference's users do
        {"name": "one_query", "kind": "one", "dtype": "int32", "dist": "lognormal", "n": 1_000_000, "nq": 16},
        # a short request against a large resident index: latency and launches
        {"name": "search_small", "kind": "search", "dtype": "int32", "dist": "lognormal", "n": 10_000_000, "nq": 4096,
         "order": "desc"},
        # the headline workload: every query's position list, 10M x 10M
        {"name": "search_large", "kind": "search", "dtype": "int32", "dist": "lognormal", "n": 10_000_000,
         "nq": 10_000_000, "order": "desc"},
        # payloads instead of positions, 64-bit coordinates, ragged sizes
        {"name": "search_values_i64", "kind": "search", "dtype": "int64", "dist": "lognormal", "n": 3_000_017,
         "nq": 1_000_003, "order": "values"},
        # uneven data: hotspots, many long intervals, a few wide queries, thousands of hits each
        {"name": "search_skewed_i64", "kind": "search", "dtype": "int64", "dist": "hotspots", "n": 20_000_000,
         "nq": 100_000, "order": "desc"},
        # counts only, a large batch
        {"name": "count_large", "kind": "count", "dtype": "int32", "dist": "lognormal", "n": 10_000_000,
         "nq": 10_000_000},
        # covered length of every query
        {"name": "coverage", "kind": "coverage", "dtype": "int32", "dist": "lognormal", "n": 1_000_000,
         "nq": 1_000_000},
        # overlap test of a batch
        {"name": "has_overlaps", "kind": "any", "dtype": "int32", "dist": "lognormal", "n": 10_000_000,
         "nq": 4_000_000},
        # building the index from unsorted device tensors with a payload
        {"name": "build", "kind": "build", "dtype": "int32", "dist": "lognormal", "n": 10_000_000, "sorted": False},
        # the batch call on host arrays: host lists out, into the caller's buffers
        {"name": "host_search", "kind": "host", "dtype": "int32", "dist": "lognormal", "n": 1_000_000, "nq": 100_003,
         "order": "vector"},
        # one server batch over 24 resident sets (one per sequence name)
        {"name": "set_table", "kind": "sets", "dtype": "int32", "dist": "lognormal", "n": 5_000_000, "nq": 200_000,
         "order": "desc"},
        # a join of two interval sets
        {"name": "intersect", "kind": "intersect", "dtype": "int32", "dist": "lognormal", "n": 1_000_000,
         "nq": 200_003},
    ]


def _log(rng, lo, hi):
    """An odd or even size, log-uniform in [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search", "search", "search", "skewed", "count", "coverage", "any", "build", "host", "one",
                       "sets", "intersect"])
    c = {"kind": kind, "dtype": rng.choice(["int32", "int64"]), "dist": "lognormal"}
    if kind == "search":
        c.update(n=_log(rng, 20_000, 10_000_000), nq=_log(rng, 64, 5_000_000),
                 order=rng.choice(["desc", "vector", "values"]))
    elif kind == "skewed":
        c.update(kind="search", dtype="int64", dist="hotspots", n=_log(rng, 1_000_000, 20_000_000),
                 nq=_log(rng, 2_000, 100_000), order=rng.choice(["desc", "vector", "values"]))
    elif kind in ("count", "any"):
        c.update(n=_log(rng, 20_000, 10_000_000), nq=_log(rng, 64, 10_000_000))
    elif kind == "coverage":
        c.update(dtype="int32", n=_log(rng, 20_000, 1_000_000), nq=_log(rng, 1_000, 1_000_000))
    elif kind == "build":
        c.update(n=_log(rng, 20_000, 10_000_000), sorted=rng.random() < 0.5)
    elif kind == "host":
        c.update(n=_log(rng, 20_000, 2_000_000), nq=_log(rng, 100, 200_000),
                 order=rng.choice(["desc", "vector", "values"]))
    elif kind == "one":
        c.update(n=_log(rng, 20_000, 10_000_000), nq=16)
    elif kind == "sets":
        c.update(dtype="int32", n=_log(rng, 200_000, 5_000_000), nq=_log(rng, 1_000, 1_000_000),
                 order=rng.choice(["desc", "vector"]))
    else:
        c.update(n=_log(rng, 20_000, 2_000_000), nq=_log(rng, 1_000, 300_000))
    return c


# ---- inputs ----------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(n, g):
    return torch.randn(n, generator=g, device="cuda", dtype=torch.float64)


def _uniform(n, g, hi):
    return (torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * hi).long()


def _lognormal(n, g, mu, sigma, lo=1, hi=1 << 62):
    return torch.exp(mu + sigma * _normal(n, g)).round().long().clamp(lo, hi)


def _starts(dist, n, g):
    span = SPAN[dist]
    s = _uniform(n, g, span)
    if dist == "hotspots":
        hot = _uniform(200, _gen(77), span)
        near = (hot[_uniform(n, g, 200)] + 5e4 * _normal(n, g)).long().clamp(0, span - 1)
        s = torch.where(torch.rand(n, generator=g, device="cuda") < 0.7, s, near)
    return s


def _mixed(n, g, share, lo, hi, rest):
    """Log-uniform lengths in [lo, hi] for a share of the items, rest elsewhere."""
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    wide = torch.exp(math.log(lo) + u * (math.log(hi) - math.log(lo))).round().long()
    return torch.where(torch.rand(n, generator=g, device="cuda") < share, wide, rest)


def _intervals(case, n, seed, by_start=False):
    g = _gen(seed)
    s = _starts(case["dist"], n, g)
    if case["dist"] == "hotspots":
        length = _mixed(n, g, 0.2, 1e5, 1e7, _lognormal(n, g, 5.0, 1.0))
    else:
        length = _lognormal(n, g, 6.0, 1.5, 1, 1_000_000)
    if by_start:
        s = torch.sort(s).values
    dt = getattr(torch, case["dtype"])
    return s.to(dt), (s + length - 1).to(dt)


def _queries(case, nq, seed):
    g = _gen(seed)
    s = _starts(case["dist"], nq, g)
    if case["dist"] == "hotspots":
        length = _mixed(nq, g, 0.01, 1e6, 1e7, _lognormal(nq, g, 5.0, 1.0))
    else:
        length = _lognormal(nq, g, 7.0, 1.0)
    dt = getattr(torch, case["dtype"])
    return s.to(dt), (s + length - 1).to(dt)


def _payload(n):
    return (torch.arange(n, device="cuda", dtype=torch.int64) * 7 % 1_000_003).to(torch.int32)


def _index(case, s, e, values=None):
    return sia.DeviceIndex(np.dtype(case["dtype"])).build(s, e, values, start_sorted=False, end_sorted=False)


def _capacity(case, hits):
    """Output slots for a batch of this case: its expected total and some room."""
    nq = case["nq"]
    return int(hits * (1.05 * nq + 16.0 * math.sqrt(nq))) + 4096


def _set_sizes(n):
    """Sizes of the resident sets: log-uniform from n / 50 to n, in a fixed shuffled order."""
    k = (np.arange(N_SETS) * 7) % N_SETS
    return [int(x) for x in np.exp(np.log(n / 50) + k / (N_SETS - 1) * np.log(50.0))]


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "build":
        s, e = _intervals(case, n, seed, by_start=case["sorted"])
        return {"case": case, "s": s, "e": e, "v": _payload(n), "ix": sia.DeviceIndex(np.dtype(case["dtype"])),
                "every": torch.arange(n, device="cuda", dtype=torch.int32),
                "out": torch.empty(n, device="cuda", dtype=torch.int32)}
    nq = case["nq"]
    st = {"case": case, "nq": nq}
    if kind == "sets":
        st["table"] = sia.SetTable(64)
        for k, m in enumerate(_set_sizes(n)):
            st["table"].put(k, _index(case, *_intervals(case, m, seed * 64 + k)))
        st["ids"] = _uniform(nq, _gen(seed + 3), N_SETS).to(torch.int32)
        st["qs"], st["qe"] = _queries(case, nq, seed + (1 << 20))
        st["plan"] = torch.empty(max(st["table"].plan_bytes(nq), 256), device="cuda", dtype=torch.uint8)
        hits = sum(_hits(case, m) for m in _set_sizes(n)) / N_SETS
        st["out"] = torch.zeros(_capacity(case, hits), dtype=torch.int32, device="cuda")
        return st
    s, e = _intervals(case, n, seed)
    st["ix"] = _index(case, s, e, _payload(n) if case.get("order") == "values" or kind == "intersect" else None)
    qs, qe = _queries(case, nq, seed + (1 << 20))
    cap = _capacity(case, _hits(case, n))
    if kind in ("host", "one"):
        st["qs"], st["qe"] = qs.cpu().numpy(), qe.cpu().numpy()
        st["off"] = np.zeros(nq + 1, np.uint64)
        st["out"] = np.zeros(cap, np.int32 if case.get("order") == "values" else np.uint32)
    else:
        st["qs"], st["qe"] = qs, qe
    if kind in ("search", "intersect"):
        st["plan"] = torch.empty(max(st["ix"].plan_bytes(nq), 256), device="cuda", dtype=torch.uint8)
        st["out"] = torch.zeros(cap, dtype=torch.int32, device="cuda")
    if kind == "intersect":
        st["data"] = _payload(nq)
        st["pieces"] = [torch.zeros(cap, dtype=dt, device="cuda") for dt in (qs.dtype, qs.dtype, torch.int32, torch.int32)]
    return st


# ---- one pass ----------------------------------------------------------------------------

class _DeviceArray:
    """A device pointer of the index as an array torch can wrap without a copy."""

    def __init__(self, ptr, n, typestr):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _copy_of(ptr, n, typestr):
    """The index's array in a tensor of its own: the next build frees the array."""
    return torch.as_tensor(_DeviceArray(ptr, n, typestr), device="cuda").clone()


def _room(buf, total):
    return buf if total <= len(buf) else torch.zeros(total, dtype=buf.dtype, device="cuda")


def _run_search(st):
    ix, nq, plan, order = st["ix"], st["nq"], st["plan"], st["case"].get("order", "vector")
    off = torch.empty(nq + 1, dtype=torch.int64, device="cuda")
    ix.plan_device(st["qs"], st["qe"], plan)
    ix.offsets_planned(plan, nq, off)
    st["out"] = out = _room(st["out"], int(off[-1].item()))
    if order == "values":
        ix.values_fill_planned(plan, nq, off, out)
    else:
        ix.fill_planned(plan, nq, off, out, order=order)
    return [off, out]


def _run_intersect(st):
    off, idx = _run_search(st)
    st["pieces"] = p = [_room(x, len(idx)) for x in st["pieces"]]
    sia._native.check(sia._native.lib.siIntersectPieces(
        st["ix"].handle, st["qs"].data_ptr(), st["qe"].data_ptr(), st["data"].data_ptr(), st["nq"], off.data_ptr(),
        idx.data_ptr(), p[0].data_ptr(), p[1].data_ptr(), p[2].data_ptr(), p[3].data_ptr(), None), "siIntersectPieces")
    return [off, idx] + p


def _run_host(st):
    order, off, total = st["case"]["order"], st["off"], ctypes.c_uint64(0)
    while True:
        out = st["out"]
        ptr = (None, out.ctypes.data) if order == "values" else (out.ctypes.data, None)
        rc = sia._native.lib.siSearchHost(
            st["ix"].handle, st["qs"].ctypes.data, st["qe"].ctypes.data, st["nq"],
            sia.SI_ORDER_VECTOR if order == "vector" else sia.SI_ORDER_DESC, off.ctypes.data, *ptr, len(out),
            ctypes.byref(total))
        if rc != sia._native.SI_ERR_CAPACITY:
            sia._native.check(rc, "siSearchHost")
            return [off, out]
        st["out"] = np.zeros(int(total.value), out.dtype)


def _run_sets(st):
    t, nq = st["table"], st["nq"]
    off = torch.empty(nq + 1, dtype=torch.int64, device="cuda")
    t.offsets_device(st["ids"], st["qs"], st["qe"], st["plan"], off)
    st["out"] = out = _room(st["out"], int(off[-1].item()))
    t.fill_device(st["plan"], nq, off, out, order=st["case"]["order"])
    return [off, out]


def _run_build(st):
    ix, n = st["ix"], st["case"]["n"]
    ix.build(st["s"], st["e"], st["v"])
    p = ix.device_arrays()
    t = "<i%d" % np.dtype(st["case"]["dtype"]).itemsize
    # the payload in sorted order, read back through the index
    sia._native.check(sia._native.lib.siGatherKeys(ix.handle, st["every"].data_ptr(), n, None, None,
                                                   st["out"].data_ptr(), None), "siGatherKeys")
    return [_copy_of(p["starts"], n, t), _copy_of(p["ends"], n, t), _copy_of(p["branch"], n, "<i4"),
            _copy_of(p["perm"], n, "<i4"), st["out"]]


def _run_one(st):
    ix, qs, qe = st["ix"], st["qs"], st["qe"]
    counts, end = np.empty(st["nq"], np.int64), 0
    for k in range(st["nq"]):
        counts[k] = ix.count(qs[k:k + 1], qe[k:k + 1])[0]
        idx = ix.search(qs[k:k + 1], qe[k:k + 1], order="vector")[1]
        if end + len(idx) > len(st["out"]):
            st["out"] = np.resize(st["out"], 2 * (end + len(idx)))
        st["out"][end:end + len(idx)] = idx
        end += len(idx)
    return [counts, st["out"]]


def run(st):
    kind = st["case"]["kind"]
    if kind == "search":
        return _run_search(st)
    if kind == "sets":
        return _run_sets(st)
    if kind == "build":
        return _run_build(st)
    if kind == "one":
        return _run_one(st)
    if kind == "host":
        return _run_host(st)
    if kind == "intersect":
        return _run_intersect(st)
    ix, nq, qs, qe = st["ix"], st["nq"], st["qs"], st["qe"]
    if kind == "count":
        out = torch.empty(nq, dtype=torch.int32, device="cuda")
        ix.count_device(qs, qe, out)
        return out
    lib, check = sia._native.lib, sia._native.check
    if kind == "coverage":
        cnt = torch.empty(nq, dtype=torch.int32, device="cuda")
        cov = torch.empty(nq, dtype=torch.int32, device="cuda")
        check(lib.siCoverage(ix.handle, qs.data_ptr(), qe.data_ptr(), nq, cnt.data_ptr(), cov.data_ptr(), None),
              "siCoverage")
        return [cnt, cov]
    out = torch.empty(nq, dtype=torch.uint8, device="cuda")
    check(lib.siHasOverlaps(ix.handle, qs.data_ptr(), qe.data_ptr(), nq, out.data_ptr(), None), "siHasOverlaps")
    return out


# ---- what a pass cannot do without ---------------------------------------------------------

def _hits(case, n):
    """Mean hits of a query over n intervals."""
    if case["dist"] == "hotspots":
        return n * 206e-6
    return n * (1242.0 + 1808.0) / SPAN["lognormal"]


def work(case):
    c = np.dtype(case["dtype"]).itemsize
    kind, n = case["kind"], case["n"]
    if kind == "build":   # coordinates and payload in; the same sorted, permutation and branch out
        return {"bytes": n * (2 * c + 4) + n * (2 * c + 4 + 4 + 4), "flops": 0}
    nq = case["nq"]
    if kind == "sets":
        sizes = _set_sizes(n)
        index, hits = sum(sizes) * 2 * c, sum(_hits(case, m) for m in sizes) / N_SETS
    else:
        index, hits = n * 2 * c, _hits(case, n)
    read = 2 * c * nq + min(index, nq * 2 * (64 + c * hits))   # queries, and the starts and ends they reach
    out = {"search": 8 * (nq + 1) + 4 * hits * nq, "sets": 8 * (nq + 1) + 4 * hits * nq,
           "host": 8 * (nq + 1) + 4 * hits * nq, "one": 4 * nq + 4 * hits * nq, "count": 4 * nq, "coverage": 8 * nq,
           "any": nq, "intersect": 4 * nq + 8 * (nq + 1) + (2 * c + 12) * hits * nq}[kind]
    return {"bytes": read + out, "flops": 0}


def exact(case, seed):
    """Counts, offsets and overlap flags from sorted coordinates; no value for the lists."""
    kind = case["kind"]
    if kind not in ("search", "count", "any", "host"):
        return None
    s, e = _intervals(case, case["n"], seed)
    qs, qe = _queries(case, case["nq"], seed + (1 << 20))
    starts = torch.sort(s).values
    last = torch.searchsorted(starts, qe, right=True)
    if kind == "any":   # the last interval (by start, then by end downwards) starting at or before the query's end
        o = torch.sort(e, descending=True, stable=True).indices
        o = o[torch.sort(s[o], stable=True).indices]
        return ((last > 0) & (e[o][(last - 1).clamp(0)] >= qs)).to(torch.uint8)
    counts = last - torch.searchsorted(torch.sort(e).values, qs)
    if kind == "count":
        return counts.to(torch.int32)
    off = torch.zeros(case["nq"] + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(counts, 0, out=off[1:])
    return [off.cpu().numpy().astype(np.uint64) if kind == "host" else off, None]
