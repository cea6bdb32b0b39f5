"""GPU parity: the HIP library against the golden vectors and the CPU oracle.

Everything here calls libsuperintervals_hip.so through its C-ABI (ctypes) and
needs a GPU.  Integer results must be bit-exact: same sorted arrays, same branch,
same counts, same index lists in the same order.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import GOLDEN_CASES, load_golden, sha

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sia():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import superintervals_amd
    return superintervals_amd


def _dev_index(sia, s, e, values=None):
    ix = sia.DeviceIndex(s.dtype)
    ix.build(s, e, values)
    return ix


def _hash(orc, off, idx):
    return orc.hash_csr(off, idx)


@pytest.mark.parametrize("name", GOLDEN_CASES)
def test_golden_build_and_queries(sia, orc, name):
    print(f"[gpu] golden {name}", flush=True)
    rec, s, e, qs, qe = load_golden(name)
    data = np.arange(s.size, dtype=np.int32)
    ix = _dev_index(sia, s, e, data)
    arr = ix.download(values=True)
    assert sha(arr["starts"], arr["ends"]) == str(rec["sorted_sha256"])
    assert sha(arr["branch"]) == str(rec["branch_sha256"])
    if "c_data_sha256" in rec:
        assert sha(arr["values"]) == str(rec["c_data_sha256"])
        assert sha(arr["perm"].astype(np.int32)) == str(rec["c_data_sha256"])
    counts = ix.count(qs, qe)
    assert np.array_equal(counts, rec["counts"])
    off, idx = ix.search(qs, qe, order="desc")
    assert np.array_equal(np.diff(off), rec["counts"].astype(np.uint64))
    hd = orc.hash_csr(off, idx)
    assert np.array_equal(hd[:rec["hash_desc_prefix"].size], rec["hash_desc_prefix"])
    assert orc.digest(hd) == int(rec["hash_desc_digest"])
    offv, idxv = ix.search(qs, qe, order="vector")
    assert np.array_equal(offv, off)
    hv = orc.hash_csr(offv, idxv)
    assert orc.digest(hv) == int(rec["hash_vec_digest"])
    lo = rec["lists_offsets"]
    for q in range(lo.size - 1):
        assert np.array_equal(idx[off[q]:off[q + 1]].astype(np.int64), rec["lists_idx"][lo[q]:lo[q + 1]])
    k = rec["upper_bound"].size
    ub = ix.upper_bound(qe[:k]).astype(np.int64)
    ub[ub == 0xFFFFFFFF] = -1
    assert np.array_equal(ub, rec["upper_bound"])
    assert np.array_equal(np.packbits(ix.has_overlaps(qs, qe)), rec["has_overlaps"])
    if "hash_cvalues_digest" in rec:
        offval, vals = ix.search(qs, qe, values=True)
        assert np.array_equal(offval, off)
        assert orc.digest(orc.hash_csr(offval, vals)) == int(rec["hash_cvalues_digest"])
        kc = rec["coverage_prefix"].shape[0]
        c, v = ix.coverage(qs[:kc], qe[:kc])
        assert np.array_equal(np.stack([c.astype(np.int64), v.astype(np.int64)], 1), rec["coverage_prefix"])
    ix.close()


@pytest.mark.parametrize("seed", range(8))
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_random_vs_oracle(sia, orc, seed, dtype):
    print(f"[gpu] random seed={seed} dtype={np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(100 + seed)
    n = int(rng.choice([1, 2, 63, 64, 65, 4095, 4096, 4097, 20_000, 150_000]))
    span = int(rng.choice([50, 5_000, 1_000_000]))
    s = rng.integers(-span, span, n).astype(dtype)
    L = rng.geometric(1.0 / max(2, span // 50), n)
    e = (s + L - 1).astype(dtype)
    if seed % 2:   # presorted input takes the no-sort path
        o = np.lexsort((-e.astype(np.int64), s.astype(np.int64)))
        s, e = s[o], e[o]
    if dtype == np.int64:
        s = s + (dtype(3) << 40)
        e = e + (dtype(3) << 40)
    nq = 30_000
    qs = rng.integers(-span - 10, span + 10, nq).astype(dtype)
    qe = (qs + rng.integers(-5, span // 20 + 5, nq)).astype(dtype)   # a few inverted
    if dtype == np.int64:
        qs = qs + (dtype(3) << 40)
        qe = qe + (dtype(3) << 40)
    oix = orc.build_index(s, e)
    ix = _dev_index(sia, s, e, np.arange(n, dtype=np.int32))
    a = ix.download(values=True)
    assert np.array_equal(a["starts"], oix["starts"]) and np.array_equal(a["ends"], oix["ends"])
    assert np.array_equal(a["branch"], oix["branch"])
    assert np.array_equal(a["values"], oix["data"])
    ocount = orc.count_batch(oix, qs, qe)
    from superintervals_amd import autotune
    saved = autotune.current()
    try:
        for cr in (0, 1):                   # the walk, and the rank form (walk for inverted queries)
            autotune.apply({"count_rank": cr})
            assert np.array_equal(ix.count(qs, qe), ocount), cr
    finally:
        autotune.apply(saved)
    for order, mode in (("desc", 0), ("vector", 1)):
        off, idx = ix.search(qs, qe, order=order)
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=mode)
        assert np.array_equal(off, ooff)
        assert np.array_equal(idx.astype(np.int64), oidx)
    off, vals = ix.search(qs, qe, values=True)
    assert np.array_equal(vals, oix["data"][orc.search_batch(oix, qs, qe, mode=0)[1]])
    ub = ix.upper_bound(qe).astype(np.int64)
    ub[ub == 0xFFFFFFFF] = -1
    assert np.array_equal(ub, np.searchsorted(oix["starts"], qe, side="right") - 1)
    ho = np.array([orc.has_overlaps(oix, x, y) for x, y in zip(qs[:3000], qe[:3000])])
    assert np.array_equal(ix.has_overlaps(qs[:3000], qe[:3000]), ho)
    if dtype == np.int32:
        c, v = ix.coverage(qs[:3000], qe[:3000])
        want = [orc.coverage(oix, x, y) for x, y in zip(qs[:3000], qe[:3000])]
        assert np.array_equal(np.stack([c, v], 1).astype(np.int64), np.array(want, np.int64))
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_upper_bound_tree_and_halving(sia, dtype):
    """Both upper_bound forms (Eytzinger top + block separators, and plain halving) against
    numpy on sizes around the 64-start blocks and the 4095-key top, long duplicate runs
    across block boundaries, and keys at the type's extremes."""
    from superintervals_amd import autotune
    info = np.iinfo(dtype)
    rng = np.random.default_rng(91)
    saved = autotune.current()
    try:
        for n in (1, 63, 64, 65, 4095 * 64, 4096 * 64 + 1, 300_001):
            for kind in range(3):
                if kind == 0:
                    s = np.sort(rng.integers(info.min, info.max, n, dtype=np.int64)).astype(dtype)
                elif kind == 1:
                    s = np.sort(rng.integers(0, max(2, n // 50), n)).astype(dtype)
                else:
                    s = np.sort(np.concatenate([rng.integers(0, 10, n // 2),
                                                np.full(n - n // 2, info.max, np.int64)])).astype(dtype)
                ix = _dev_index(sia, s, s)
                st = ix.download()["starts"]
                xs = np.concatenate([st[rng.integers(0, n, 500)].astype(np.int64),
                                     st[rng.integers(0, n, 200)].astype(np.int64) - 1,
                                     st[rng.integers(0, n, 200)].astype(np.int64) + 1,
                                     [info.min, info.max, int(st[0]) - 1],
                                     rng.integers(info.min, info.max, 300, dtype=np.int64)])
                xs = np.clip(xs, info.min, info.max).astype(dtype)
                want = np.searchsorted(st, xs, side="right").astype(np.int64) - 1
                for tree in (1, 0):
                    autotune.apply({"ub_tree": tree})
                    got = ix.upper_bound(xs).astype(np.int64)
                    got[got == 0xFFFFFFFF] = -1
                    assert np.array_equal(got, want), (n, kind, tree)
                ix.close()
    finally:
        autotune.apply(saved)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_search_keys_and_items(sia, orc, dtype):
    """Batched search_keys / search_items (superintervals.hpp:913-971): the descending walk's
    hits as (start, end) and (start, end, value), against the oracle's descending lists."""
    print(f"[gpu] search_keys/items dtype={np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(77)
    n = 30_000
    s = rng.integers(0, 2_000_000, n).astype(dtype)
    e = (s + rng.geometric(1 / 400, n) - 1).astype(dtype)
    if dtype == np.int64:
        s, e = s + (dtype(5) << 36), e + (dtype(5) << 36)
    vals = rng.integers(-2**31, 2**31 - 1, n).astype(np.int32)
    qs = rng.integers(0, 2_000_000, 20_000).astype(dtype)
    qe = (qs + rng.integers(0, 3_000, qs.size)).astype(dtype)
    if dtype == np.int64:
        qs, qe = qs + (dtype(5) << 36), qe + (dtype(5) << 36)
    ix = _dev_index(sia, s, e, vals)
    oix = orc.build_index(s, e, vals)
    ooff, oidx = orc.search_batch(oix, qs, qe, mode=0)
    off, ks, ke = ix.search_keys(qs, qe)
    assert np.array_equal(off, ooff.astype(np.uint64))
    assert np.array_equal(ks.astype(np.int64), oix["starts"][oidx].astype(np.int64))
    assert np.array_equal(ke.astype(np.int64), oix["ends"][oidx].astype(np.int64))
    off2, ks2, ke2, kv2 = ix.search_keys(qs, qe, items=True)
    assert np.array_equal(off2, off) and np.array_equal(ks2, ks) and np.array_equal(ke2, ke)
    assert np.array_equal(kv2, oix["data"][oidx])
    off0, ks0, ke0 = ix.search_keys(qs[:0], qe[:0])
    assert off0.tolist() == [0] and ks0.size == 0
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_planned_batch_reuse(sia, orc, dtype):
    """One plan serves count, offsets and every fill mode, repeatedly, on one stream."""
    import torch
    print(f"[gpu] planned reuse dtype={np.dtype(dtype).name}", flush=True)
    rec, s, e, qs, qe = load_golden("c1_shuffled")
    s, e, qs, qe = (x.astype(dtype) for x in (s, e, qs, qe))
    ix = _dev_index(sia, s, e, np.arange(s.size, dtype=np.int32))
    oix = orc.build_index(s, e)
    dev = torch.device("cuda:0")
    tqs, tqe = torch.from_numpy(qs).to(dev), torch.from_numpy(qe).to(dev)
    nq = qs.size
    plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device=dev)
    ix.plan_device(tqs, tqe, plan)
    counts = torch.empty(nq, dtype=torch.int32, device=dev)
    off = torch.empty(nq + 1, dtype=torch.int64, device=dev)
    for _ in range(2):
        ix.count_planned(plan, nq, counts)
        assert np.array_equal(counts.cpu().numpy().astype(np.uint32), rec["counts"])
        ix.offsets_planned(plan, nq, off, counts)
        assert np.array_equal(np.diff(off.cpu().numpy()), rec["counts"].astype(np.int64))
    total = int(off[-1].item())
    idx = torch.empty(total, dtype=torch.int32, device=dev)
    offh = off.cpu().numpy().astype(np.uint64)
    for order, key in (("desc", "hash_desc_digest"), ("vector", "hash_vec_digest"), ("desc", "hash_desc_digest")):
        idx.fill_(-7)
        ix.fill_planned(plan, nq, off, idx, order=order)
        h = orc.hash_csr(offh, idx.cpu().numpy().view(np.uint32))
        assert orc.digest(h) == int(rec[key]), order
    vals = torch.empty(total, dtype=torch.int32, device=dev)
    ix.values_fill_planned(plan, nq, off, vals)
    ooff, oidx = orc.search_batch(oix, qs, qe, mode=0)
    assert np.array_equal(vals.cpu().numpy(), oix["data"][oidx])
    ix.close()


def test_launch_choices_do_not_change_results(sia, orc):
    """Every tile size / residency choice the autotuner may pick gives identical output."""
    from superintervals_amd import autotune
    rec, s, e, qs, qe = load_golden("c2_1m")
    ix = _dev_index(sia, s, e)
    saved = autotune.current()
    try:
        for tile, cw, fw, cr, orank, psl, rs in ((64, 1, 1, 0, 1, 0, 1), (512, 0, 1, 1, 0, 1, 0),
                                                 (4096, 1, 0, 1, 1, 2, 1), (100000, 0, 0, 0, 0, 1, 0),
                                                 (1024, 0, 0, 1, 1, 2, 1), (1024, 0, 0, 0, 0, 0, 0)):
            print(f"[gpu] launch tile={tile} count_wgs={cw} fill_wgs={fw} rank={cr}/{orank} skip_low={psl} "
                  f"range_skip={rs}", flush=True)
            autotune.apply({"tile": tile, "count_wgs": cw, "fill_wgs": fw, "count_rank": cr,
                            "offsets_rank": orank, "plan_skip_low": psl, "range_skip": rs})
            assert np.array_equal(ix.count(qs, qe), rec["counts"])
            off, idx = ix.search(qs, qe, order="vector")
            assert orc.digest(orc.hash_csr(off, idx)) == int(rec["hash_vec_digest"])
    finally:
        autotune.apply(saved)
    with pytest.raises(sia.SIError):
        autotune.apply({"tile": 3})
    ix.close()


@pytest.mark.parametrize("lane_steps", [1, 3, 17])
def test_heavy_path_parity(sia, orc, lane_steps):
    """Walks parked after lane_steps lines finish in the wave-cooperative kernel with the
    same results, in every mode (count by walk, descending, vector, values)."""
    from superintervals_amd import autotune
    print(f"[gpu] heavy path lane_steps={lane_steps}", flush=True)
    rec, s, e, qs, qe = load_golden("c1_shuffled")
    ix = _dev_index(sia, s, e, np.arange(s.size, dtype=np.int32))
    oix = orc.build_index(s, e)
    saved = autotune.current()
    try:
        autotune.apply({"lane_steps": lane_steps, "offsets_rank": 0, "count_rank": 0})
        assert np.array_equal(ix.count(qs, qe), rec["counts"])
        off, idx = ix.search(qs, qe, order="desc")
        assert orc.digest(orc.hash_csr(off, idx)) == int(rec["hash_desc_digest"])
        off, idx = ix.search(qs, qe, order="vector")
        assert orc.digest(orc.hash_csr(off, idx)) == int(rec["hash_vec_digest"])
        off, vals = ix.search(qs, qe, values=True)
        assert orc.digest(orc.hash_csr(off, vals)) == int(rec["hash_cvalues_digest"])
    finally:
        autotune.apply(saved)
    ix.close()


@pytest.mark.parametrize("lane_steps,far", [(1, False), (40, False), (1, True)])
def test_heavy_path_int64_long_walks(sia, orc, lane_steps, far):
    """int64 hotspot mixture (workload 3 distributions): every walk parked after lane_steps
    lines and finished by the wave-cooperative kernel, which fetches four lines at a time
    and leaves a line through exitp lookups.  Ends within 2^32 of each other are read from
    the 32-bit copy; far = True adds intervals 2^40 away, so the index has no such copy.
    Counts, both orders and values equal the oracle's."""
    from superintervals_amd import autotune
    print(f"[gpu] heavy path int64 lane_steps={lane_steps} far={far}", flush=True)
    s, e = sia.workload_intervals(3, 1_000_000, seed=33, sorted=False)
    if far:
        extra = (np.int64(1) << 40) + np.arange(0, 2000 * 97, 97, dtype=np.int64)
        s = np.concatenate([s, extra])
        e = np.concatenate([e, extra + 500])
    qs, qe = sia.workload_queries(3, 6_000, seed=34)
    # ragged edges: queries before, after and around the whole index, and a point query
    qs = np.concatenate([qs, np.array([-5, 0, int(e.max()), int(s.min()), 10**9], np.int64)])
    qe = np.concatenate([qe, np.array([-1, int(e.max()) + 10, int(e.max()) + 10, int(s.min()), 10**9], np.int64)])
    vals = (np.arange(s.size, dtype=np.int64) * 7 % 1_000_003).astype(np.int32)
    ix = _dev_index(sia, s, e, vals)
    oix = orc.build_index(s, e, vals)
    saved = autotune.current()
    try:
        autotune.apply({"lane_steps": lane_steps, "offsets_rank": 0, "count_rank": 0})
        ocounts = orc.count_batch(oix, qs, qe)
        assert np.array_equal(ix.count(qs, qe), ocounts)
        for order, mode in (("desc", 0), ("vector", 1)):
            off, idx = ix.search(qs, qe, order=order)
            ooff, oidx = orc.search_batch(oix, qs, qe, mode=mode)
            assert np.array_equal(off, ooff), order
            assert np.array_equal(idx.astype(np.int64), oidx), order
        off, v = ix.search(qs, qe, values=True)
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=0)
        assert np.array_equal(v, oix["data"][oidx])
        # a walk with more than 4 x 64 hits spans more lines than one fetch holds
        assert (ocounts > 4 * 64).sum() > 100
    finally:
        autotune.apply(saved)
    ix.close()


def test_autotune_picks_and_keeps_results(sia, orc):
    """tune() on a planned batch picks tile, residency, lane step budget and count form,
    applies them, and the library's output with them equals the oracle's."""
    import torch
    from superintervals_amd import autotune
    print("[gpu] autotune on workload 3 (300K int64 intervals)", flush=True)
    s, e = sia.workload_intervals(3, 300_000, seed=35, sorted=False)
    qs, qe = sia.workload_queries(3, 4_000, seed=36)
    ix = _dev_index(sia, s, e)
    oix = orc.build_index(s, e)
    dev = torch.device("cuda:0")
    tqs, tqe = torch.from_numpy(qs).to(dev), torch.from_numpy(qe).to(dev)
    nq = qs.size
    plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device=dev)
    off = torch.empty(nq + 1, dtype=torch.int64, device=dev)
    saved = autotune.current()
    try:
        ix.plan_device(tqs, tqe, plan)
        ix.offsets_planned(plan, nq, off)
        total = int(off[-1].item())
        idx = torch.empty(max(total, 1), dtype=torch.int32, device=dev)
        best, table = autotune.tune(ix, plan, nq, off, idx, reps=1, tiles=(512, 2048), wgs=(0,),
                                    lane_steps=(16, 256), qs_t=tqs, qe_t=tqe)
        assert best["lane_steps"] in (16, 256) and best["count_rank"] in (0, 1)
        assert best["plan_sync"] in (0, 1) and best["plan_skip_low"] in (0, 1)
        now = autotune.current()
        for k, v in autotune.knobs_of(best).items():
            assert now[k] == v, k
        assert len(table) == 2 + 2 + 2 + 2 + 2
        # the plan redone during tuning is still this batch's plan
        ix.offsets_planned(plan, nq, off)
        ix.fill_planned(plan, nq, off, idx, order="desc")
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=0)
        assert np.array_equal(off.cpu().numpy().astype(np.uint64), ooff)
        assert np.array_equal(idx[:total].cpu().numpy().view(np.uint32).astype(np.int64), oidx)
        counts = ix.count(qs, qe)
        assert np.array_equal(counts, orc.count_batch(oix, qs, qe))
        o, i = ix.search(qs, qe, order="desc")
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=0)
        assert np.array_equal(o, ooff) and np.array_equal(i.astype(np.int64), oidx)
    finally:
        autotune.apply(saved)
    ix.close()


def test_workload3_wide_queries(sia, orc):
    """int64 hotspot mixture with 1 % wide queries (workload 3 distributions, 2M intervals),
    unsorted input: full CSR against the oracle in both orders."""
    print("[gpu] workload 3 (2M int64 intervals, 20K queries)", flush=True)
    s, e = sia.workload_intervals(3, 2_000_000, seed=31, sorted=False)
    qs, qe = sia.workload_queries(3, 20_000, seed=32)
    ix = _dev_index(sia, s, e, np.arange(s.size, dtype=np.int32))
    oix = orc.build_index(s, e)
    a = ix.download(values=True)
    assert np.array_equal(a["starts"], oix["starts"]) and np.array_equal(a["branch"], oix["branch"])
    assert np.array_equal(a["values"], oix["data"])
    counts = ix.count(qs, qe)
    ocounts = orc.count_batch(oix, qs, qe)
    assert np.array_equal(counts, ocounts)
    assert ocounts.max() > 5_000           # the wide queries exceed the lane step budget
    for order, mode in (("desc", 0), ("vector", 1)):
        off, idx = ix.search(qs, qe, order=order)
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=mode)
        assert np.array_equal(off, ooff)
        assert np.array_equal(idx.astype(np.int64), oidx)
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_wide_queries_guaranteed_run(sia, orc, dtype):
    """Queries much wider than the intervals: most hits are the run [lower_bound(s),
    upper_bound(e)] taken without reading ends.  Every mode and order, the run taken or
    walked, lane and wave walks, against the oracle; some runs reach position 0."""
    from superintervals_amd import autotune
    print(f"[gpu] wide queries, guaranteed run dtype={np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(77)
    n = 150_000
    s = rng.integers(0, 3_000_000, n)
    e = s + rng.integers(0, 200, n)
    long_ = rng.random(n) < 0.02
    e = np.where(long_, s + rng.integers(1000, 200_000, n), e)
    qs = rng.integers(-5_000, 3_000_000, 6000)
    qe = qs + rng.integers(20_000, 400_000, qs.size)
    qs[:50] = -10                        # runs that reach position 0
    base = (np.int64(9) << 34) if dtype == np.int64 else 0
    s, e, qs, qe = ((x + base).astype(dtype) for x in (s, e, qs, qe))
    ix = _dev_index(sia, s, e, np.arange(n, dtype=np.int32))
    oix = orc.build_index(s, e)
    ocount = orc.count_batch(oix, qs, qe)
    st = oix["starts"]
    run = np.searchsorted(st, qe, side="right") - np.searchsorted(st, qs, side="left")
    assert run.sum() > 0.8 * ocount.sum()      # the run dominates
    want = {o: orc.search_batch(oix, qs, qe, mode=m) for o, m in (("desc", 0), ("vector", 1))}
    saved = autotune.current()
    try:
        for rs in (1, 0):
            for ls in (1024, 2):
                autotune.apply({"range_skip": rs, "lane_steps": ls, "count_rank": 0, "offsets_rank": 0})
                assert np.array_equal(ix.count(qs, qe), ocount), (rs, ls)
                for order in ("desc", "vector"):
                    off, idx = ix.search(qs, qe, order=order)
                    assert np.array_equal(off, want[order][0]) and np.array_equal(idx.astype(np.int64), want[order][1]), (rs, ls, order)
                off, vals = ix.search(qs, qe, values=True)
                assert np.array_equal(vals, oix["data"][want["desc"][1]])
    finally:
        autotune.apply(saved)
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_range_lengths_around_wave_written_threshold(sia, orc, dtype):
    """Range segments of 64 or more values are written by the whole wave, shorter ones in
    the shared 64-slot chunks.  Runs of exactly 1..1000 values (63, 64, 65, 127, 128, 129
    among them), next to line masks from a few longer intervals, in every mode and order,
    against the oracle."""
    print(f"[gpu] range lengths around the wave-written threshold dtype={np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(5)
    n = 100_000
    s = np.arange(n, dtype=np.int64)
    e = s + 1
    longer = rng.random(n) < 0.05
    e = np.where(longer, s + rng.integers(2, 300, n), e)
    lens = np.array([1, 2, 31, 32, 33, 63, 64, 65, 66, 127, 128, 129, 191, 192, 193, 1000])
    L = np.repeat(lens, 300)
    qs = rng.integers(0, n - 1200, L.size)
    qe = qs + L - 1
    base = (np.int64(5) << 33) if dtype == np.int64 else 0
    s, e, qs, qe = ((x + base).astype(dtype) for x in (s, e, qs, qe))
    ix = _dev_index(sia, s, e, np.arange(n, dtype=np.int32))
    oix = orc.build_index(s, e)
    assert np.array_equal(ix.count(qs, qe), orc.count_batch(oix, qs, qe))
    for order, mode in (("desc", 0), ("vector", 1)):
        off, idx = ix.search(qs, qe, order=order)
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=mode)
        assert np.array_equal(off, ooff) and np.array_equal(idx.astype(np.int64), oidx), order
    off, vals = ix.search(qs, qe, values=True)
    ooff, oidx = orc.search_batch(oix, qs, qe, mode=0)
    assert np.array_equal(vals, oix["data"][oidx])
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_plan_sort_forms_order_queries_by_end(sia, dtype):
    """The plan sorts the queries by end, stably.  Both forms of its radix sort (plan_sync
    1: a host read-back of the digit histograms skips the digits that are equal for every
    query; 0: every digit is sorted, with no read-back) must give numpy's stable argsort of
    the ends, for one item, one tile, a partial last tile and thousands of tiles, with ends
    that are random, spread over the whole coordinate range, few distinct values (long runs
    of equal digits, and digits constant over the batch), runs of equal ends (digit counts
    taken once per wave where a wave's digits agree, per lane elsewhere) or all equal (the
    read-back form then runs no pass)."""
    import torch
    from superintervals_amd import autotune
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(91)
    s, e = sia.workload_intervals(2, 100_000, seed=92, sorted=True)
    ix = _dev_index(sia, s.astype(dtype), e.astype(dtype))
    info = np.iinfo(dtype)
    saved = autotune.current()
    try:
        for nq in (1, 2, 2047, 2048, 2049, 65_537, 3_000_001):
            for kind in ("random", "wide", "few", "runs", "equal"):
                print(f"[gpu] plan sort dtype={np.dtype(dtype).name} nq={nq} ends={kind}", flush=True)
                if kind == "random":
                    qe = rng.integers(0, 2_000_000, nq)
                elif kind == "wide":
                    qe = rng.integers(info.min // 2, info.max // 2, nq)
                elif kind == "few":
                    qe = rng.choice(np.array([-3, 0, 255, 256, 70_000], dtype=np.int64), nq)
                elif kind == "runs":   # runs of ~100 equal ends: most waves see one digit value
                    qe = np.repeat(rng.integers(-5_000_000, 5_000_000, nq // 100 + 1), 100)[:nq]
                else:   # every digit constant: the read-back form runs no pass
                    qe = np.full(nq, 12_345, dtype=np.int64)
                qe = qe.astype(dtype)
                qs = (qe.astype(np.int64) - rng.integers(0, 1000, nq)).astype(dtype)
                want = np.argsort(qe, kind="stable")
                tqs, tqe = torch.from_numpy(qs).to(dev), torch.from_numpy(qe).to(dev)
                plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device=dev)
                for ps in (1, 0):
                    autotune.apply({"plan_sync": ps, "plan_skip_low": 0})
                    plan.fill_(0xA5)
                    ix.plan_device(tqs, tqe, plan)
                    torch.cuda.synchronize()
                    q = plan[256:256 + 4 * nq].view(torch.int32).cpu().numpy()
                    assert np.array_equal(q, want), (nq, kind, ps)
    finally:
        autotune.apply(saved)
    ix.close()


@pytest.mark.parametrize("dtype,long_len", [(np.int64, 0), (np.int64, 4096), (np.int32, 64), (np.int32, 1)])
def test_long_list_walk(sia, orc, dtype, long_len):
    """The wave walk with a long list: hits below the first start >= s - len come from the
    list of intervals longer than len.  Built with the threshold chosen from the lengths
    (0) or forced, queries on the wave walk (lane_steps 2) and not, the list used or not,
    every mode and order against the oracle."""
    from superintervals_amd import autotune
    print(f"[gpu] long list dtype={np.dtype(dtype).name} long_len={long_len}", flush=True)
    if dtype == np.int64:
        s, e = sia.workload_intervals(3, 2_000_000, seed=33, sorted=False)
        qs, qe = sia.workload_queries(3, 6000, seed=34)
    else:
        rng = np.random.default_rng(12)
        n = 300_000
        s = rng.integers(0, 20_000_000, n)
        e = s + np.where(rng.random(n) < 0.1, rng.integers(5000, 2_000_000, n), rng.integers(-3, 300, n))
        qs = rng.integers(0, 20_000_000, 6000)
        qe = qs + rng.integers(-2, 3000, qs.size)
        s, e, qs, qe = (x.astype(np.int32) for x in (s, e, qs, qe))
    saved = autotune.current()
    try:
        autotune.apply({"long_len": long_len})
        ix = _dev_index(sia, s, e, np.arange(s.size, dtype=np.int32))
    finally:
        autotune.apply(saved)
    oix = orc.build_index(s, e)
    wc = orc.count_batch(oix, qs, qe)
    want = {o: orc.search_batch(oix, qs, qe, mode=m) for o, m in (("desc", 0), ("vector", 1))}
    try:
        for lw in (1, 0):
            for ls in (2, 1024):
                autotune.apply({"long_walk": lw, "lane_steps": ls, "count_rank": 0, "offsets_rank": 0})
                assert np.array_equal(ix.count(qs, qe), wc), (lw, ls)
                for order in ("desc", "vector"):
                    off, idx = ix.search(qs, qe, order=order)
                    assert np.array_equal(off, want[order][0]), (lw, ls, order)
                    assert np.array_equal(idx.astype(np.int64), want[order][1]), (lw, ls, order)
                off, vals = ix.search(qs, qe, values=True)
                assert np.array_equal(vals, oix["data"][want["desc"][1]]), (lw, ls)
        # single queries take the wave walk with the list too
        autotune.apply({"long_walk": 1})
        for q in range(0, 200, 7):
            assert ix.count(qs[q:q + 1], qe[q:q + 1])[0] == wc[q]
            off, idx = ix.search(qs[q:q + 1], qe[q:q + 1], order="vector")
            assert np.array_equal(idx.astype(np.int64), orc.search(oix, qs[q], qe[q], 1))
    finally:
        autotune.apply(saved)
    ix.close()


def test_learned_index(sia, orc):
    """Learned upper_bound (workload 4 distributions, 2M intervals): GPU gradients against the
    float64 oracle, output identical to the plain search, and the trained root's gain over the
    untrained (identity-CDF) one in leaf corrections."""
    import torch
    from oracle import rmi
    print("[gpu] learned index", flush=True)
    s, e = sia.workload_intervals(4, 2_000_000, seed=41, sorted=False)
    ix = _dev_index(sia, s, e)
    starts = ix.download()["starts"]
    n = starts.size
    dev = torch.device("cuda:0")

    untrained = sia.LearnedIndex(ix, 4096)
    info0 = untrained.train(steps=0)
    model = sia.LearnedIndex(ix, 4096)
    info1 = model.train(steps=400, batch=65536, lr=3e-3)
    assert info1["loss"] < 1e-3

    # gradients of the training kernels against the oracle, at the initial and trained points
    kmin, inv = model.norm()
    pos = np.random.default_rng(3).integers(0, n, 4096).astype(np.uint32)
    x = (np.float64(starts[pos].astype(np.int64) - kmin) * np.float64(np.float32(inv))).astype(np.float32)
    t = (pos.astype(np.float32) / np.float32(n)).astype(np.float32)
    for p in (rmi.identity_params().astype(np.float32), model.params()):
        g_gpu = model.gradient(pos, p)
        g_cpu, l_cpu = rmi.gradient(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
        scale = np.abs(g_cpu).max()
        assert np.all(np.abs(g_gpu[:-1] - g_cpu) <= 1e-4 * scale + 2e-3 * np.abs(g_cpu)), \
            np.abs(g_gpu[:-1] - g_cpu).max() / scale
        assert abs(g_gpu[-1] - l_cpu) <= 1e-5 + 1e-3 * l_cpu

    # identical to the plain upper_bound on point, short-range and out-of-range queries
    qs, qe = sia.workload_queries(4, 1_000_000, seed=42)
    xs = np.concatenate([qe, qs, starts[:1000], starts[-1000:], np.array([np.iinfo(np.int32).min,
                         np.iinfo(np.int32).max, int(starts[0]) - 1, int(starts[-1]) + 1], np.int32)])
    xt = torch.from_numpy(xs).to(dev)
    plain = torch.empty(xs.size, dtype=torch.int32, device=dev)
    assert sia._native.lib.siUpperBound(ix.handle, xt.data_ptr(), xs.size, plain.data_ptr(), None) == 0
    want = np.searchsorted(starts, xs, side="right").astype(np.int64) - 1
    got_plain = plain.cpu().numpy().view(np.uint32).astype(np.int64)
    got_plain[got_plain == 0xFFFFFFFF] = -1
    assert np.array_equal(got_plain, want)
    corr = {}
    for name, m in (("untrained", untrained), ("trained", model)):
        out = torch.empty(xs.size, dtype=torch.int32, device=dev)
        st = torch.zeros(3, dtype=torch.int64, device=dev)
        m.upper_bound_device(xt, out, st)
        got = out.cpu().numpy().view(np.uint32).astype(np.int64)
        got[got == 0xFFFFFFFF] = -1
        assert np.array_equal(got, want), name
        fb, w, c = st.cpu().tolist()
        corr[name] = c / xs.size
        print(f"[gpu] {name}: fallbacks {fb}, mean window {w / xs.size:.1f}, mean leaf correction "
              f"{c / xs.size:.2f}", flush=True)
    # Leaves own fixed position ranges, so the windows do not depend on the root; what the
    # trained network gains is naming the right leaf: fewer correction steps than the
    # identity-CDF root on a density that varies 100x between segments.
    print(f"[gpu] max leaf error bound {info1['max_abs_err']}", flush=True)
    assert info0["max_abs_err"] == info1["max_abs_err"]
    assert corr["trained"] < 0.25 * corr["untrained"]
    model.close()
    untrained.close()
    ix.close()


def test_learned_plan_forms_and_forced_fallback(sia, orc):
    """The learned model as the plan's bound search (knob ub_learned): the batched search and
    count through it equal the plain-halving and tree forms and the oracle.  With every leaf
    window narrowed (test knob learned_shrink) the queries take the whole-leaf fallback and
    the output is still identical.  A rebuilt index drops the model; destroying the index
    before the model is safe."""
    import torch
    from superintervals_amd import autotune
    print("[gpu] learned plan forms and forced fallback", flush=True)
    s, e = sia.workload_intervals(4, 1_000_000, seed=43, sorted=False)
    ix = _dev_index(sia, s, e)
    model = sia.LearnedIndex(ix, 4096)
    model.train(steps=200, batch=65536, lr=3e-3)
    qs, qe = sia.workload_queries(4, 200_000, seed=44)
    qs[:100] = np.iinfo(np.int32).min          # lower bound of the smallest value
    oix = orc.build_index(s, e)
    wd = orc.search_batch(oix, qs, qe, mode=0)
    wv = orc.search_batch(oix, qs, qe, mode=1)
    wc = orc.count_batch(oix, qs, qe)
    saved = autotune.current()
    try:
        for knobs in ({"ub_tree": 0, "ub_learned": 0}, {"ub_tree": 1, "ub_learned": 0}, {"ub_learned": 1},
                      {"ub_learned": 1, "range_skip": 0}, {"ub_learned": 1, "learned_shrink": 1 << 20},
                      {"ub_learned": 1, "learned_shrink": 3}):
            autotune.apply(dict({"ub_tree": 1, "range_skip": 1, "learned_shrink": 0}, **knobs))
            print(f"[gpu] plan bounds {knobs}", flush=True)
            assert np.array_equal(ix.count(qs, qe), wc), knobs
            off, idx = ix.search(qs, qe, order="desc")
            assert np.array_equal(off, wd[0]) and np.array_equal(idx.astype(np.int64), wd[1]), knobs
            off, idx = ix.search(qs, qe, order="vector")
            assert np.array_equal(off, wv[0]) and np.array_equal(idx.astype(np.int64), wv[1]), knobs
        # the forced fallback, counted: identical to upper_bound with fallbacks > 0
        starts = ix.download()["starts"]
        want = np.searchsorted(starts, qe, side="right").astype(np.int64) - 1
        xt = torch.from_numpy(qe).cuda()
        for shrink in (0, 3, 1 << 20):
            autotune.apply({"learned_shrink": shrink})
            out = torch.empty(qe.size, dtype=torch.int32, device="cuda")
            st = torch.zeros(3, dtype=torch.int64, device="cuda")
            model.upper_bound_device(xt, out, st)
            got = out.cpu().numpy().view(np.uint32).astype(np.int64)
            got[got == 0xFFFFFFFF] = -1
            assert np.array_equal(got, want), shrink
            fb = int(st[0].item())
            print(f"[gpu] learned_shrink {shrink}: fallbacks {fb}", flush=True)
            if shrink == 0:
                assert fb == 0
            if shrink == 1 << 20:
                assert fb >= int((want >= 0).sum())    # every query with a position took it
    finally:
        autotune.apply(saved)
    # rebuilding the index drops the model: ub_learned then plans through the tree
    ix.build(s, e)
    with pytest.raises(sia.SIError):
        model.upper_bound_device(xt, torch.empty(qe.size, dtype=torch.int32, device="cuda"))
    try:
        autotune.apply({"ub_learned": 1})
        assert np.array_equal(ix.count(qs, qe), wc)
    finally:
        autotune.apply(saved)
    ix.close()                   # the index first: the model forgets it
    model.close()


def test_walk_stats_match_oracle(sia, orc):
    import torch
    rec, s, e, qs, qe = load_golden("c1_sorted")
    ix = _dev_index(sia, s, e)
    tot = ix.walk_stats_device(torch.from_numpy(qs).cuda(), torch.from_numpy(qe).cuda())
    oix = orc.build_index(s, e)
    h, v, j = orc.walk_stats_batch(oix, qs, qe)
    assert tot[:3] == [h, v, j]
    assert tot[0] == int(rec["counts"].sum())


def test_empty_and_edge_cases(sia, orc):
    # empty index: every query is well defined and finds nothing
    ix = sia.DeviceIndex(np.int32).build(np.zeros(0, np.int32), np.zeros(0, np.int32))
    q = np.array([1, 5], np.int32)
    assert ix.count(q, q).tolist() == [0, 0]
    off, idx = ix.search(q, q)
    assert off.tolist() == [0, 0, 0] and idx.size == 0
    assert ix.has_overlaps(q, q).tolist() == [False, False]
    # empty query batch
    ix1 = sia.DeviceIndex(np.int32).build(np.array([1], np.int32), np.array([10], np.int32))
    assert ix1.count(np.zeros(0, np.int32), np.zeros(0, np.int32)).size == 0
    off, idx = ix1.search(np.zeros(0, np.int32), np.zeros(0, np.int32))
    assert off.tolist() == [0] and idx.size == 0
    assert ix1.count([1, 11], [5, 20]).tolist() == [1, 0]
    # int32 extremes
    big, small = np.iinfo(np.int32).max, np.iinfo(np.int32).min
    s = np.array([small, small, 0, big - 5, big], np.int32)
    e = np.array([small, big, 10, big, big], np.int32)
    qs = np.array([small, small, 5, big, big, 0, big], np.int32)
    qe = np.array([small, big, 5, big, big - 1, small, small], np.int32)
    ixe = sia.DeviceIndex(np.int32).build(s, e)
    oix = orc.build_index(s, e)
    assert np.array_equal(ixe.count(qs, qe), orc.count_batch(oix, qs, qe))
    # the rank form (#{ends < s} through the sorted-ends tree; s = min has none below) at
    # both widths' extremes, for count and for the offsets of a search
    from superintervals_amd import autotune
    saved = autotune.current()
    try:
        for dt in (np.int32, np.int64):
            lo, hi = np.iinfo(dt).min, np.iinfo(dt).max
            s2 = np.array([lo, lo, 0, hi - 5, hi, lo + 1], dt)
            e2 = np.array([lo, hi, 10, hi, hi, lo + 1], dt)
            qs2 = np.array([lo, lo, 5, hi, hi, 0, hi, lo + 1, lo], dt)
            qe2 = np.array([lo, hi, 5, hi, hi - 1, lo, lo, lo + 1, lo + 1], dt)
            ix2 = sia.DeviceIndex(dt).build(s2, e2)
            oix2 = orc.build_index(s2, e2)
            want = orc.count_batch(oix2, qs2, qe2)
            for ub_tree in (1, 0):
                autotune.apply({"count_rank": 1, "offsets_rank": 1, "ub_tree": ub_tree})
                assert np.array_equal(ix2.count(qs2, qe2), want), (dt, ub_tree)
                off, idx = ix2.search(qs2, qe2)
                ooff, oidx = orc.search_batch(oix2, qs2, qe2, mode=0)
                assert np.array_equal(off, ooff) and np.array_equal(idx.astype(np.int64), oidx), (dt, ub_tree)
            ix2.close()
    finally:
        autotune.apply(saved)
    # query before build
    with pytest.raises(sia.SIError):
        sia.DeviceIndex(np.int32).count(q, q)


def _capi():
    import superintervals_amd._native as N
    return N


def test_capi_reference_functions(sia, orc):
    """The reference C-ABI (c_superintervals.h names) on the device index."""
    N = _capi()
    L = N.lib
    rec, s, e, qs, qe = load_golden("c1_shuffled")
    h = L.createSuperIntervals()
    L.reserveSuperIntervals(h, 16)
    for i in range(s.size):
        L.addInterval(h, int(s[i]), int(e[i]), i)
    st = N.cSuperIntervals.from_address(h)
    assert st.size == s.size and not st.startSorted
    L.indexSuperIntervals(h)
    st = N.cSuperIntervals.from_address(h)
    assert st.startSorted and st.endSorted and st.idx == 0
    n = s.size
    hs = np.ctypeslib.as_array(st.starts, (n,)).copy()
    he = np.ctypeslib.as_array(st.ends, (n,)).copy()
    hd = np.ctypeslib.as_array(st.data, (n,)).copy()
    hb = np.ctypeslib.as_array(st.branch, (n,)).copy().view(np.int64)
    assert sha(hs, he) == str(rec["sorted_sha256"])
    assert sha(hb) == str(rec["branch_sha256"])
    assert sha(hd) == str(rec["c_data_sha256"])
    oix = orc.build_index(s, e)
    res = N.cIndexResult()
    for q in range(0, 300):
        a, b = int(qs[q]), int(qe[q])
        assert L.countOverlaps(h, a, b) == rec["counts"][q]
        L.clearIndexResult(C.byref(res))
        L.searchIdxs(h, a, b, C.byref(res))
        got = [res.data[k] for k in range(res.size)]
        assert got == orc.search(oix, a, b, 0).tolist()
        L.clearIndexResult(C.byref(res))
        L.searchValues(h, a, b, C.byref(res))
        assert [res.data[k] for k in range(res.size)] == orc.values(oix, a, b).tolist()
        ub = L.upperBound(h, b)
        want = orc.upper_bound(oix, b)
        assert (ub == 2 ** 64 - 1 and want == -1) or ub == want
        assert N.cSuperIntervals.from_address(h).idx == ub
        assert L.anyOverlaps(h, a, b) == orc.has_overlaps(oix, a, b)
        cnt = C.c_size_t(0)
        cov = C.c_int32(0)
        L.coverage(h, a, b, C.byref(cnt), C.byref(cov))
        assert (cnt.value, cov.value) == orc.coverage(oix, a, b)
    # appending semantics: results accumulate until cleared (c_superintervals.h:209-210)
    L.clearIndexResult(C.byref(res))
    L.searchIdxs(h, int(qs[0]), int(qe[0]), C.byref(res))
    L.searchIdxs(h, int(qs[1]), int(qe[1]), C.byref(res))
    assert res.size == rec["counts"][0] + rec["counts"][1]
    L.destroyIndexResult(C.byref(res))
    keys = N.cKeyResult()
    items = N.cItemResult()
    L.searchKeys(h, int(qs[5]), int(qe[5]), C.byref(keys))
    L.searchItems(h, int(qs[5]), int(qe[5]), C.byref(items))
    strict = orc.search(oix, qs[5], qe[5], 0)
    assert [(keys.data[k].start, keys.data[k].end) for k in range(keys.size)] == \
        [(int(oix["starts"][j]), int(oix["ends"][j])) for j in strict]
    assert [items.data[k].data for k in range(items.size)] == [int(oix["data"][j]) for j in strict]
    L.destroyKeyResult(C.byref(keys))
    L.destroyItemResult(C.byref(items))
    # batch extensions
    counts = np.empty(qs.size, np.uint32)
    assert L.siCountBatch(h, qs.ctypes.data, qe.ctypes.data, qs.size, counts.ctypes.data) == 0
    assert np.array_equal(counts, rec["counts"])
    off = np.empty(qs.size + 1, np.uint64)
    tot = C.c_uint64(0)
    rc = L.siSearchIdxsBatch(h, qs.ctypes.data, qe.ctypes.data, qs.size, off.ctypes.data, None, 0, C.byref(tot))
    assert rc == N.SI_ERR_CAPACITY and tot.value == int(rec["counts"].sum())
    idx = np.empty(tot.value, np.int32)
    assert L.siSearchIdxsBatch(h, qs.ctypes.data, qe.ctypes.data, qs.size, off.ctypes.data, idx.ctypes.data,
                               idx.size, C.byref(tot)) == 0
    assert orc.digest(orc.hash_csr(off, idx.astype(np.int64))) == int(rec["hash_desc_digest"])
    vals = np.empty(tot.value, np.int32)
    assert L.siSearchValuesBatch(h, qs.ctypes.data, qe.ctypes.data, qs.size, off.ctypes.data,
                                 vals.ctypes.data, vals.size, C.byref(tot)) == 0
    assert orc.digest(orc.hash_csr(off, vals)) == int(rec["hash_cvalues_digest"])
    L.destroySuperIntervals(h)


def test_capi_empty_and_unindexed(sia):
    N = _capi()
    L = N.lib
    h = L.createSuperIntervals()
    L.indexSuperIntervals(h)              # empty: no-op, as the reference
    assert L.countOverlaps(h, 1, 5) == 0
    assert not L.anyOverlaps(h, 1, 5)
    L.addInterval(h, 1, 10, 7)
    assert L.countOverlaps(h, 1, 5) == 0   # not indexed yet: no result, error recorded
    assert b"indexSuperIntervals" in L.siGetLastError()
    L.indexSuperIntervals(h)
    assert L.countOverlaps(h, 1, 5) == 1 and L.countOverlaps(h, 11, 20) == 0
    L.destroySuperIntervals(h)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_single_query_path(sia, orc, dtype):
    """One-query host calls run one wave on the index's scratch: every mode against the
    batched path and the oracle, repeated calls (the capacity probe), a result larger than
    the scratch (the batched path takes it), an index with start > end intervals."""
    import superintervals_amd._native as N
    print(f"[gpu] single-query path dtype={np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(8)
    n = 300_000
    s = rng.integers(0, 3_000_000, n)
    e = s + rng.geometric(1 / 200, n) - 1
    inv = rng.random(n) < 0.01
    base = (np.int64(5) << 33) if dtype == np.int64 else 0
    for with_inv in (False, True):
        ee = np.where(inv, s - 3, e) if with_inv else e
        ss_, ee_ = (s + base).astype(dtype), (ee + base).astype(dtype)
        ix = _dev_index(sia, ss_, ee_, np.arange(n, dtype=np.int32))
        oix = orc.build_index(ss_, ee_)
        qs = rng.integers(-10, 3_000_000, 400)
        qe = qs + rng.integers(0, 5000, qs.size)
        qe[::13] = qs[::13] - 2                                  # inverted queries
        qs[0], qe[0] = 0, 3_000_000                               # every interval: > 65536 results
        qs, qe = (qs + base).astype(dtype), (qe + base).astype(dtype)
        for q in range(qs.size):
            a, b = qs[q:q + 1], qe[q:q + 1]
            assert ix.count(a, b)[0] == orc.count(oix, a[0], b[0])
            for order, mode in (("desc", 0), ("vector", 1)):
                off, idx = ix.search(a, b, order=order)   # probe + fill: the second call reuses the first
                assert np.array_equal(idx.astype(np.int64), orc.search(oix, a[0], b[0], mode)), (q, order)
            off, vals = ix.search(a, b, values=True)
            assert np.array_equal(vals, oix["data"][orc.search(oix, a[0], b[0], 0)])
            ub = int(ix.upper_bound(b)[0])
            want = orc.upper_bound(oix, b[0])
            assert (ub == 0xFFFFFFFF and want == -1) or ub == want
            assert bool(ix.has_overlaps(a, b)[0]) == orc.has_overlaps(oix, a[0], b[0])
        # capacity probe through the C-ABI-style call: too small, then exact, both right
        tot = C.c_uint64(0)
        o2 = np.zeros(2, np.uint64)
        small = np.zeros(1, np.uint32)
        a, b = qs[5:6], qe[5:6]
        want = orc.search(oix, a[0], b[0], 0)
        if want.size > 1:
            rc = N.lib.siSearchHost(ix.handle, a.ctypes.data, b.ctypes.data, 1, 0, o2.ctypes.data, small.ctypes.data,
                                    None, 1, C.byref(tot))
            assert rc == N.SI_ERR_CAPACITY and tot.value == want.size and o2[1] == want.size
            big = np.zeros(want.size, np.uint32)
            assert N.lib.siSearchHost(ix.handle, a.ctypes.data, b.ctypes.data, 1, 0, o2.ctypes.data, big.ctypes.data,
                                      None, big.size, C.byref(tot)) == 0
            assert np.array_equal(big.astype(np.int64), want)
        ix.close()


def test_capi_stale_handle_after_clear_and_add(sia):
    """A handle changed after indexSuperIntervals has no device index until it is indexed
    again, even when the new contents have the old size."""
    N = _capi()
    L = N.lib
    h = L.createSuperIntervals()
    for s0, e0 in [(1, 10), (5, 20), (30, 40)]:
        L.addInterval(h, s0, e0, 0)
    L.indexSuperIntervals(h)
    assert L.countOverlaps(h, 8, 9) == 2
    L.clearSuperIntervals(h)
    for s0, e0 in [(100, 110), (105, 120), (130, 140)]:
        L.addInterval(h, s0, e0, 0)
    assert L.countOverlaps(h, 8, 9) == 0 and L.countOverlaps(h, 106, 107) == 0
    assert b"indexSuperIntervals" in L.siGetLastError()
    L.indexSuperIntervals(h)
    assert L.countOverlaps(h, 106, 107) == 2 and L.countOverlaps(h, 8, 9) == 0
    L.addInterval(h, 1, 500, 0)           # one more after indexing: stale again
    assert L.countOverlaps(h, 106, 107) == 0
    L.indexSuperIntervals(h)
    assert L.countOverlaps(h, 106, 107) == 3
    L.destroySuperIntervals(h)


def _extras():
    import os
    from conftest import GOLDEN
    return dict(np.load(os.path.join(GOLDEN, "extras.npz")))


@pytest.mark.parametrize("lane_steps", [256, 2])
def test_index_with_inverted_intervals_golden(sia, orc, lane_steps):
    """An index in which 15 % of the intervals have start > end: every count form and both
    orders against the reference's outputs (the rank forms are not exact there, so the
    library walks)."""
    from superintervals_amd import autotune
    print(f"[gpu] inverted intervals lane_steps={lane_steps}", flush=True)
    x = _extras()
    s, e, qs, qe = x["inv_starts"], x["inv_ends"], x["inv_qs"], x["inv_qe"]
    ix = _dev_index(sia, s, e, np.arange(s.size, dtype=np.int32))
    saved = autotune.current()
    try:
        autotune.apply({"lane_steps": lane_steps})
        for cr in (0, 1):
            for orank in (0, 1):
                autotune.apply({"count_rank": cr, "offsets_rank": orank})
                assert np.array_equal(ix.count(qs, qe).astype(np.int64), x["inv_counts"]), (cr, orank)
                off, idx = ix.search(qs, qe, order="desc")
                assert np.array_equal(off, x["inv_desc_off"]) and np.array_equal(idx.astype(np.int32), x["inv_desc_idx"])
                off, idx = ix.search(qs, qe, order="vector")
                assert np.array_equal(off, x["inv_vec_off"]) and np.array_equal(idx.astype(np.int32), x["inv_vec_idx"])
                off, vals = ix.search(qs, qe, values=True)
                assert np.array_equal(off, x["inv_cval_off"]) and np.array_equal(vals, x["inv_cval"])
    finally:
        autotune.apply(saved)
    ix.close()
    # the C-ABI on the same intervals
    N = _capi()
    L = N.lib
    h = L.createSuperIntervals()
    for i in range(s.size):
        L.addInterval(h, int(s[i]), int(e[i]), i)
    L.indexSuperIntervals(h)
    res = N.cIndexResult()
    off = x["inv_cidx_off"].astype(np.int64)
    for q in range(0, qs.size, 7):
        L.clearIndexResult(C.byref(res))
        L.searchIdxs(h, int(qs[q]), int(qe[q]), C.byref(res))
        assert [res.data[k] for k in range(res.size)] == x["inv_cidx"][off[q]:off[q + 1]].tolist()
        assert L.countOverlaps(h, int(qs[q]), int(qe[q])) == x["inv_counts"][q]
    L.destroyIndexResult(C.byref(res))
    L.destroySuperIntervals(h)


@pytest.mark.parametrize("order", ["desc", "vector"])
def test_fill_reports_offsets_that_disagree(sia, orc, order):
    """A fill never writes outside a query's segment; with offsets that disagree with the
    index (one query given a slot too many, or one too few) siPlanCheck reports it."""
    import torch
    N = _capi()
    print(f"[gpu] fill/offsets mismatch order={order}", flush=True)
    rng = np.random.default_rng(5)
    s = np.sort(rng.integers(0, 100_000, 20_000)).astype(np.int32)
    e = (s + rng.integers(0, 500, s.size)).astype(np.int32)
    qs = rng.integers(0, 100_000, 5000).astype(np.int32)
    qe = (qs + rng.integers(0, 300, qs.size)).astype(np.int32)
    ix = _dev_index(sia, s, e)
    dev = torch.device("cuda:0")
    tqs, tqe = torch.from_numpy(qs).to(dev), torch.from_numpy(qe).to(dev)
    nq = qs.size
    plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device=dev)
    off = torch.empty(nq + 1, dtype=torch.int64, device=dev)
    ix.plan_device(tqs, tqe, plan)
    ix.offsets_planned(plan, nq, off)
    torch.cuda.synchronize()
    counts = np.diff(off.cpu().numpy())
    q = int(np.flatnonzero(counts >= 2)[0])
    total = int(off[-1].item())
    idx = torch.full((total + 1,), -1, dtype=torch.int32, device=dev)
    ix.fill_planned(plan, nq, off, idx, order=order)
    assert N.lib.siPlanCheck(ix.handle, plan.data_ptr(), None) == N.SI_OK
    ref = idx[:total].clone()
    # query q given one slot too many: its list leaves a gap
    bad = off.clone()
    bad[q + 1:] += 1
    idx.fill_(-1)
    ix.fill_planned(plan, nq, bad, idx, order=order)
    assert N.lib.siPlanCheck(ix.handle, plan.data_ptr(), None) == N.SI_ERR_MISMATCH
    # query q given one slot too few (q + 1 one more): q's list is cut, never overrun
    bad = off.clone()
    bad[q + 1] -= 1
    idx.fill_(-1)
    ix.fill_planned(plan, nq, bad, idx, order=order)
    assert N.lib.siPlanCheck(ix.handle, plan.data_ptr(), None) == N.SI_ERR_MISMATCH
    o0, o1 = int(off[q].item()), int(off[q + 1].item())
    assert torch.equal(idx[o0:o1 - 1], ref[o0:o1 - 1])
    # and a correct fill clears the report
    ix.fill_planned(plan, nq, off, idx, order=order)
    assert N.lib.siPlanCheck(ix.handle, plan.data_ptr(), None) == N.SI_OK
    assert torch.equal(idx[:total], ref)
    ix.close()


def test_python_intervalmap_mirror(sia, orc):
    """The Python IntervalMap mirrors intervalmap.pyx on the reference's examples."""
    m = sia.IntervalMap()
    for s, e, v in [(10, 20, "a"), (11, 12, None), (13, 14, None), (15, 16, None), (25, 29, "d")]:
        m.add(s, e, v)
    m.build()
    assert m.has_overlaps(17, 30) and not m.has_overlaps(1, 3)
    assert m.search_values(17, 30) == ["d", "a"]
    assert m.count(17, 30) == 2
    assert m.search_idxs(17, 30) == [4, 0]
    assert m.coverage(10, 29)[1] == 17
    m2 = sia.IntervalMap.from_arrays([1, 2, 4, 5, 6, 60], [100, 3, 50, 50, 50, 70])
    assert m2.search_idxs(10, 65) == [2, 3, 4, 5, 0]          # vector order (pyx uses it)
    assert [x.tolist() for x in m2.search_idxs_batch([10, 1], [65, 1])] == [[2, 3, 4, 5, 0], [0]]
    assert m2.count_batch([10, 200], [65, 300]).tolist() == [5, 0]
    with pytest.raises(ValueError):
        m2.count_batch([1, 2], [3])


def test_cpp_api_program(sia):
    """include/superintervals.hpp (si::IntervalMap<S, T>) through a compiled C++ program."""
    import os
    import subprocess
    from conftest import ROOT
    exe = os.path.join(ROOT, "tests", "cpp", "test_intervalmap")
    assert os.path.exists(exe), "build the C++ test first (__graft_entry__.build())"
    print("[gpu] C++ API program", flush=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


@pytest.mark.parametrize("knobs", [None, {"tile": 512, "count_wgs": 0, "fill_wgs": 0, "lane_steps": 1024,
                                          "count_rank": 1, "plan_sync": 0, "plan_skip_low": 1}],
                         ids=["defaults", "benched"])
def test_full_size_lognormal_10Mx10M_properties(sia, orc, knobs):
    """10M intervals x 10M queries (log-normal lengths): size-independent properties of the whole
    output plus an oracle check of a query sample, with the library's default launch choices
    and with those the headline benchmark's autotuner picks (512-query tiles, no plan
    read-back, the lowest end digit unsorted)."""
    import torch
    from superintervals_amd import autotune
    print(f"[gpu] full-size log-normal 10M x 10M knobs={knobs}", flush=True)
    saved = autotune.current()
    if knobs:
        autotune.apply(knobs)
    try:
        _full_size_lognormal(sia, orc)
    finally:
        autotune.apply(saved)


def _full_size_lognormal(sia, orc):
    import torch
    n = nq = 10_000_000
    s, e = sia.workload_intervals(2, n, seed=1, sorted=True)
    qs, qe = sia.workload_queries(2, nq, seed=2)
    ix = _dev_index(sia, s, e)
    dev = torch.device("cuda:0")
    tqs, tqe = torch.from_numpy(qs).to(dev), torch.from_numpy(qe).to(dev)
    off = torch.empty(nq + 1, dtype=torch.int64, device=dev)
    counts = torch.empty(nq, dtype=torch.int32, device=dev)
    ix.offsets_device(tqs, tqe, off, counts)
    torch.cuda.synchronize()
    total = int(off[-1].item())
    # closed form: count = #starts <= e - #ends < s (all queries have s <= e)
    ss = torch.from_numpy(s).to(dev)
    se = torch.sort(torch.from_numpy(e).to(dev)).values
    closed = torch.searchsorted(ss, tqe, right=True) - torch.searchsorted(se, tqs, right=False)
    assert torch.equal(closed.to(torch.int32), counts)
    assert torch.equal(off[1:] - off[:-1], counts.to(torch.int64))
    idx = torch.empty(max(total, 1), dtype=torch.int32, device=dev)
    ix.fill_device(tqs, tqe, off, idx, order="desc")
    torch.cuda.synchronize()
    d = ix.device_arrays()
    ends_t = torch.from_numpy(ix.download()["ends"]).to(dev)
    starts_t = ss
    # every emitted position overlaps its query
    qid = torch.repeat_interleave(torch.arange(nq, device=dev), counts.to(torch.int64))
    pos = idx[:total].to(torch.int64)
    assert bool((starts_t[pos] <= tqe[qid]).all()) and bool((ends_t[pos] >= tqs[qid]).all())
    # strictly descending inside every list
    same = qid[1:] == qid[:-1]
    assert bool((pos[1:][same] < pos[:-1][same]).all())
    # oracle on a sample
    oix = orc.build_index(s, e)
    sample = np.arange(0, nq, 4999)
    ooff, oidx = orc.search_batch(oix, qs[sample], qe[sample], mode=0)
    offh = off.cpu().numpy().astype(np.uint64)
    idxh = idx[:total].cpu().numpy()
    for k, q in enumerate(sample):
        assert np.array_equal(idxh[offh[q]:offh[q + 1]].astype(np.int64), oidx[ooff[k]:ooff[k + 1]])
    del d
    ix.close()


def test_output_offsets_beyond_2_31(sia):
    """Lists whose output offsets pass 2^31 entries (8.7 GB of positions) on n = 2^24 + 5
    intervals [i, n + i], with queries in triples: [0, n - 1] hits all n as one guaranteed
    run longer than 2^23 (written on its own by the whole wave), [0, 2^21 - 1] hits 2^21 as
    a run of whole 64-slot chunks, and the point 2^23, whose 2^23 hits below its run are
    walked by the wave-cooperative kernel.  Both orders; every entry is checked against the
    closed form."""
    import torch
    print("[gpu] output offsets beyond 2^31", flush=True)
    n, r2, p3, trip = (1 << 24) + 5, 1 << 21, 1 << 23, 80
    s = np.arange(n, dtype=np.int32)
    e = (s + n).astype(np.int32)
    ix = _dev_index(sia, s, e)
    qs = np.zeros(3 * trip, np.int32)
    qe = np.tile(np.array([n - 1, r2 - 1, p3], np.int32), trip)
    qs[2::3] = p3
    dev = torch.device("cuda:0")
    tqs, tqe = torch.from_numpy(qs).to(dev), torch.from_numpy(qe).to(dev)
    off = torch.empty(qs.size + 1, dtype=torch.int64, device=dev)
    ix.offsets_device(tqs, tqe, off)
    torch.cuda.synchronize()
    per = n + r2 + p3 + 1
    total = int(off[-1].item())
    assert total == trip * per and total > (1 << 31)
    idx = torch.empty(total, dtype=torch.int32, device=dev)
    rows = idx.view(trip, per)
    desc = torch.cat([torch.arange(n - 1, -1, -1), torch.arange(r2 - 1, -1, -1), torch.arange(p3, -1, -1)])
    vec = torch.cat([torch.arange(n), torch.arange(r2), torch.arange(p3 + 1)])
    for order, row in (("desc", desc), ("vector", vec)):
        idx.fill_(-1)
        ix.fill_device(tqs, tqe, off, idx, order=order)
        torch.cuda.synchronize()
        assert bool((rows == row.to(torch.int32).to(dev)).all()), order
    del rows, idx
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n,nq,depth", [(1, 3, 1), (63, 64, 5), (64, 65, 64), (129, 257, 130), (5000, 1, 255),
                                        (5000, 1023, 256), (5000, 1025, 257), (70_000, 70_001, 40),
                                        (300_000, 4096, 300), (40_000, 300_000, 600), (100_000, 400_000, 1),
                                        (3000, 400_000, 3)])
def test_sweep_fill(sia, orc, dtype, n, nq, depth):
    """The fill's sweep over query starts: lists of about `depth` intervals holding a point
    (255, 256, 257 and more: around and past what the sweep keeps in registers), batches that
    give a wave one query, part of a register and several, starts close together, in clusters
    far apart and at the ends of the coordinate range, queries with start > end, and queries
    past every interval; both orders and the values equal the oracle's."""
    print(f"[gpu] sweep fill dtype={np.dtype(dtype).name} n={n} nq={nq} depth={depth}", flush=True)
    rng = np.random.default_rng(n + nq + depth)
    info = np.iinfo(dtype)
    step = 7
    s = np.sort(rng.integers(0, step * n + 1, n))
    # lengths: exactly depth / step positions for most, a few long ones, a stretch of dense starts
    e = s + np.where(rng.random(n) < 0.02, rng.integers(1, 50 * step * depth + 2, n), rng.integers(1, 2 * step * depth + 2, n))
    e[: n // 50] += step * n // 3
    qs = rng.integers(-50, step * n + 500, nq)
    far = rng.random(nq)
    qs = np.where(far < 0.05, rng.integers(step * n // 2, step * n // 2 + 40, nq), qs)
    qe = qs + np.where(rng.random(nq) < 0.9, rng.integers(0, 40 * step, nq), rng.integers(-30 * step, 200 * step, nq))
    qs[-1], qe[-1] = info.min, info.max
    qs[0] = info.min if nq > 1 else qs[0]
    if nq > 3:
        qs[1], qe[1] = info.max, info.max
        qs[2], qe[2] = info.max, info.min
    s, e, qs, qe = (x.astype(dtype) for x in (s, e, qs, qe))
    vals = (np.arange(n, dtype=np.int64) * 7 % 1_000_003).astype(np.int32)
    ix = _dev_index(sia, s, e, vals)
    oix = orc.build_index(s, e, vals)
    for order, mode in (("desc", 0), ("vector", 1)):
        off, idx = ix.search(qs, qe, order=order)
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=mode)
        assert np.array_equal(off, ooff) and np.array_equal(idx.astype(np.int64), oidx), order
    off, v = ix.search(qs, qe, values=True)
    ooff, oidx = orc.search_batch(oix, qs, qe, mode=0)
    assert np.array_equal(v, oix["data"][oidx])
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n", [1, 2, 3, 64, 2047, 2048, 2049, 300_001])
def test_build_finds_add_flags(sia, orc, dtype, n):
    """The build finds the add() flags of intervals in the given order (on the device) as
    add_flags does on the host: sorted inputs, one break or one rising tie at the first, the last
    and a middle place, a tie after a break (which the flags do not see), extreme coordinates,
    host arrays and device tensors; the permutation equals that of a build given add_flags'."""
    import torch
    print(f"[gpu] add flags dtype={np.dtype(dtype).name} n={n}", flush=True)
    rng = np.random.default_rng(n)
    info = np.iinfo(dtype)
    s0 = np.sort(rng.integers(0, 4 * n, n)).astype(dtype)
    e0 = (s0 + rng.integers(0, 50, n)).astype(dtype)
    o = np.lexsort((-e0.astype(np.int64), s0))
    s0, e0 = s0[o], e0[o]
    cases = [(s0, e0)]
    for k in sorted({0, n // 2, n - 2} & set(range(n - 1))):
        s, e = s0.copy(), e0.copy()
        s[k] = info.max                      # a break after k
        cases.append((s, e))
        s, e = s0.copy(), e0.copy()
        s[k + 1:] = np.maximum(s[k + 1:], s[k] + 5)
        s[k + 1] = s[k]
        e[k], e[k + 1] = info.min, info.max  # a rising tie at k
        cases.append((s, e))
        s2 = s.copy()
        s2[0] = info.max                     # the same after a break at 0
        cases.append((s2, e))
    ix, ref = sia.DeviceIndex(dtype), sia.DeviceIndex(dtype)
    for s, e in cases:
        ss, es = sia.add_flags(s, e) if dtype == np.int32 else (
            bool((s[1:] >= s[:-1]).all()), _end_sorted(s, e))
        want = ref.build(s, e, None, ss, es).download()
        ts, te = torch.from_numpy(s).cuda(), torch.from_numpy(e).cuda()
        for a, b in ((s, e), (ts, te)):
            got = ix.build(a, b).download()
            assert all(np.array_equal(got[k], want[k]) for k in ("starts", "ends", "perm", "branch"))
        assert np.array_equal(ix.build(ts, te, None, start_sorted=ss).download()["perm"], want["perm"])
    ix.close()
    ref.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("first", [0, 2046, 2047, 2048, 100_000])
def test_build_flags_with_breaks_everywhere(sia, orc, dtype, first):
    """Flags found while many workgroups report breaks and others leave because of them: sorted up
    to the first break, then in random order (every workgroup from there on holds breaks and rising
    ties), with a rising tie before the break or none; arrays as the oracle builds them."""
    print(f"[gpu] add flags, breaks from {first} dtype={np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(first)
    n = 1_000_000
    s = rng.integers(0, n // 4, n)
    e = s + rng.integers(0, 60, n)
    o = np.lexsort((-e[:first + 1], s[:first + 1]))
    s[:first + 1], e[:first + 1] = s[:first + 1][o], e[:first + 1][o]
    s[first + 1] = s[first] - 1
    s, e = s.astype(dtype), e.astype(dtype)
    ix = sia.DeviceIndex(dtype)
    for tie in (False, True):
        if tie and first > 1:
            s[1], e[1] = s[0], e[0] + 1
        got = ix.build(s, e).download()
        want = orc.build_index(s, e, np.arange(n, dtype=np.int32))
        for key in ("starts", "ends", "branch"):
            assert np.array_equal(got[key], want[key]), (tie, key)
        assert np.array_equal(got["perm"], want["data"]), tie
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n", [17, 1000, 70_001])
def test_build_with_a_wrong_promise(sia, dtype, n):
    """A build told that unsorted starts are sorted stays within its arrays and keeps the order it
    was given.  One start is out of place (larger than all, at the front, in the middle, or across
    a group of 16), so that every search bound on one side of it is still well defined; count,
    upper_bound, has_overlaps, coverage and both orders there equal a scan of the given arrays,
    for one query and for a batch."""
    print(f"[gpu] wrong promise dtype={np.dtype(dtype).name} n={n}", flush=True)
    rng = np.random.default_rng(n)
    for place in (0, 15, 16, n // 2):
        s = np.sort(rng.integers(1000, 1000 + 8 * n, n))
        e = s + rng.integers(0, 90, n)
        high = 1000 + 9 * n
        s[place], e[place] = high, high + 5
        # searches by a value x agree on the order where all keys <= x precede the others
        lo, hi = (high, high + 200) if place == 0 else (900, s[place - 1])
        qs = rng.integers(lo + 1, hi + 1, 40)
        qe = np.minimum(qs + rng.integers(0, 60, 40), hi)
        s, e, qs, qe = (x.astype(dtype) for x in (s, e, qs, qe))
        ix = sia.DeviceIndex(dtype).build(s, e, None, start_sorted=True, end_sorted=True)
        got = ix.download()
        assert np.array_equal(got["starts"], s) and np.array_equal(got["ends"], e)
        hits = [np.flatnonzero((s <= b) & (e >= a))[::-1] for a, b in zip(qs, qe)]
        ub = np.array([np.flatnonzero(s <= b).max(initial=-1) for b in qe])
        one = [(slice(k, k + 1), hits[k:k + 1]) for k in range(5)]
        for at, want in [(slice(0, 40), hits)] + one:
            a, b = qs[at], qe[at]
            assert np.array_equal(ix.count(a, b), [len(h) for h in want])
            assert np.array_equal(ix.upper_bound(b).view(np.int32), ub[at])
            any_ = (ub[at] >= 0) & (e[np.maximum(ub[at], 0)] >= a)
            assert np.array_equal(ix.has_overlaps(a, b), any_)
            off, idx = ix.search(a, b)
            assert np.array_equal(off, np.concatenate([[0], np.cumsum([len(h) for h in want])]))
            assert np.array_equal(idx.astype(np.int64), np.concatenate(want))
            if dtype == np.int32:
                c, v = ix.coverage(a, b)
                cov = [int((np.minimum(e[h], y) - np.maximum(s[h], x)).sum()) for h, x, y in zip(want, a, b)]
                assert np.array_equal(c, [len(h) for h in want]) and np.array_equal(v, cov)
        ix.close()


def _end_sorted(s, e):
    """add()'s end flag by comparisons (add_flags subtracts, which wraps at the int64 limits)."""
    for k in range(s.size - 1):
        if s[k + 1] < s[k]:
            return True
        if s[k + 1] == s[k] and e[k + 1] > e[k]:
            return False
    return True


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 255, 256, 257, 4097, 70_001])
def test_build_shapes_of_ends(sia, orc, dtype, n):
    """The build against the oracle (sorted arrays, permutation, branch, payload) at the edges of
    the 16-ary max tree's groups and levels, for ends that rise (every branch open to the left,
    none found), fall (each branch the neighbour), are equal, saw-tooth over groups, reach back
    to one far position, hold the type's extremes, and for starts in runs of equal values: of up
    to 32 (mended in place) and longer (sorted by both coordinates), all equal, with equal pairs;
    presorted or not."""
    print(f"[gpu] build shapes dtype={np.dtype(dtype).name} n={n}", flush=True)
    rng = np.random.default_rng(n)
    info = np.iinfo(dtype)
    i = np.arange(n, dtype=np.int64)
    shapes = {
        "rising": (i * 3, i * 3 + 1), "falling": (i, 2 * n - i), "equal ends": (i, np.full(n, n)),
        "saw": (i, i + (16 - i % 16) * 5), "back": (i, np.where(i == n // 3, 10 * n, i)),
        "runs": (i // 32, rng.integers(0, 40, n)), "runs of 33": (i // 33, rng.integers(0, 40, n)),
        "one start": (np.zeros(n, np.int64), rng.integers(0, 10, n)),
        "pairs": (rng.integers(0, n // 4 + 1, n), rng.integers(-5, 5, n)),
        "random": (rng.integers(0, 10 * n, n), rng.integers(0, 10 * n, n)),
    }
    ends = np.array([info.min, info.max, info.max - 1, info.min + 1, 0], dtype=np.int64)
    shapes["extremes"] = (rng.choice(ends, n), rng.choice(ends, n))
    from superintervals_amd import autotune
    ix = sia.DeviceIndex(dtype)
    saved = autotune.current()
    try:
        for name, (s, e) in shapes.items():
            for shuffled in (False, True):
                o = rng.permutation(n) if shuffled else i
                a, b = s[o].astype(dtype), e[o].astype(dtype)
                autotune.apply(saved)
                got = ix.build(a, b, i.astype(np.int32)).download(values=True)
                want = orc.build_index(a, b, i.astype(np.int32))
                for key in ("starts", "ends", "branch"):
                    assert np.array_equal(got[key], want[key]), (name, shuffled, key)
                assert np.array_equal(got["values"], want["data"]), (name, shuffled)
                assert np.array_equal(got["perm"], want["data"]), (name, shuffled)
                # the line walk reads the exits
                q = np.concatenate([a[:50], b[:50], rng.integers(0, 10 * n, 50).astype(dtype)])
                autotune.apply({"count_rank": 0, "range_skip": 0})
                assert np.array_equal(ix.count(q, q), orc.count_batch(want, q, q)), (name, shuffled)
    finally:
        autotune.apply(saved)
    ix.close()


def test_builds_from_threads_keep_their_blocks(sia, orc):
    """Indexes built, rebuilt (larger, smaller, empty) and destroyed from several threads at once,
    on streams of their own: every index stays what its own intervals give (the device blocks
    that builds pass on to one another never serve two at a time)."""
    import threading
    import torch
    print("[gpu] builds from threads", flush=True)
    errors = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            st = torch.cuda.Stream()
            live = []
            for k, n in enumerate((70_000, 500, 90_000, 0, 66_000, 120_000)):
                s = rng.integers(0, 1_000_000, n).astype(np.int32)
                e = (s + rng.integers(0, 3000, n)).astype(np.int32)
                ix = live.pop()[0] if k % 2 and live else sia.DeviceIndex(np.int32)
                live.append((ix.build(s, e, stream=st), orc.build_index(s, e)))
                for a, want in live:
                    got = a.download()
                    for key in ("starts", "ends", "branch"):
                        assert np.array_equal(got[key], want[key]), (seed, k, key)
            for a, _ in live:
                a.close()
        except BaseException as x:   # noqa: B902
            errors.append(x)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nq", [2048 * 127 + 1, 2048 * 128, 2048 * 128 + 1])
def test_plan_sort_around_the_scan_free_size(sia, dtype, nq):
    """The plan's sort at the batch size from which its passes scan the tiles' digit counts with
    kernels of their own (above 128 tiles of 2048): numpy's stable argsort of the ends, for ends
    over the whole range, with one digit that varies, and none."""
    import torch
    print(f"[gpu] plan sort dtype={np.dtype(dtype).name} nq={nq}", flush=True)
    rng = np.random.default_rng(nq)
    info = np.iinfo(dtype)
    ix = _dev_index(sia, np.arange(1000, dtype=dtype), np.arange(1000, dtype=dtype) + 5)
    for qe in (rng.integers(info.min, info.max, nq), 7 + 256 * rng.integers(0, 256, nq), np.full(nq, -1)):
        qe = qe.astype(dtype)
        t = torch.from_numpy(qe).cuda()
        plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device="cuda")
        ix.plan_device(t, t, plan)
        torch.cuda.synchronize()
        q = plan[256:256 + 4 * nq].view(torch.int32).cpu().numpy()
        assert np.array_equal(q, np.argsort(qe, kind="stable"))
    ix.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 4095, 4096, 4097, 70_003])
@pytest.mark.parametrize("inverted", [False, True])
def test_coverage(sia, orc, n, inverted):
    """Count and covered length against the oracle around the sizes of lines and tree nodes, with
    coordinates over the whole int32 range (the sums wrap), equal starts and ends, queries with
    s > e, s = e, at both ends of the range and beyond all intervals, and with intervals of
    start > end in the index (the walk)."""
    print(f"[gpu] coverage n={n} inverted={inverted}", flush=True)
    rng = np.random.default_rng(n)
    info = np.iinfo(np.int32)
    for wide in (False, True):
        lo, hi = (info.min, info.max) if wide else (-1000, 10 * n)
        s = rng.integers(lo, hi, n)
        length = rng.integers(0, (hi - lo) // 8 if wide else 300, n)
        e = np.minimum(s + length, info.max)
        s[: n // 4], e[: n // 4] = s[0], e[0]
        if inverted:
            s[-1], e[-1] = e[-1], s[-1] - 1 if s[-1] > info.min else s[-1]
        s, e = s.astype(np.int32), e.astype(np.int32)
        qs = np.concatenate([rng.integers(lo, hi, 400), s[:100], e[:100], [info.min, info.min, info.max, 0]])
        qe = np.concatenate([qs[:400] + rng.integers(-50, 3000, 400), s[:100], e[:100] + 0, [info.min, info.max, info.max, -1]])
        qe = np.clip(qe, info.min, info.max)
        qs, qe = qs.astype(np.int32), qe.astype(np.int32)
        ix = _dev_index(sia, s, e)
        oix = orc.build_index(s, e)
        c, v = ix.coverage(qs, qe)
        want = [orc.coverage(oix, a, b) for a, b in zip(qs, qe)]
        assert np.array_equal(c.astype(np.int64), [w[0] for w in want])
        assert np.array_equal(v.astype(np.int64), [w[1] for w in want])
        ix.close()


@pytest.mark.parametrize("shape", ["even", "gap", "crowd", "one point", "wide"])
@pytest.mark.parametrize("n", [1, 4, 15, 17, 4096, 20_011])
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_bucket_tables(sia, orc, dtype, n, shape):
    """upper_bound, count and has_overlaps through the bucket tables: buckets of one key, of up to
    16 and of more, empty buckets in runs longer than a wave fills (a far interval), tables given
    up because most keys share a bucket, all keys equal, and coordinates over the whole range of
    the type."""
    print(f"[gpu] bucket tables {np.dtype(dtype).name} n={n} {shape}", flush=True)
    rng = np.random.default_rng(n)
    info = np.iinfo(dtype)
    if shape == "wide":
        s = rng.integers(info.min, info.max, n, dtype=dtype)
        e = np.maximum(s, rng.integers(info.min, info.max, n, dtype=dtype))
        s[0], e[-1] = info.min, info.max
    else:
        s = rng.integers(0, 1 if shape == "one point" else 9 * n, n).astype(dtype)
        e = (s + (0 if shape == "one point" else rng.integers(0, 200, n))).astype(dtype)
        if shape == "gap":
            s[-1], e[-1] = 900 * n, 900 * n + 10
        elif shape == "crowd":
            s[-1], e[-1] = 2**30, 2**30 + 1
    ix = _dev_index(sia, s, e)
    oix = orc.build_index(s, e)
    near = rng.integers(-3, 4, 200)
    at = np.concatenate([s[rng.integers(0, n, 100)], e[rng.integers(0, n, 100)]]).astype(object) + near
    any_ = rng.integers(info.min, info.max, 100, dtype=dtype).astype(object)
    qs = np.concatenate([at, any_, [info.min, info.min, info.max, info.max, 0]])
    qe = np.concatenate([at + rng.integers(-5, 300, 200), any_[::-1], [info.min, info.max, info.max, info.min, 0]])
    qs = np.clip(qs, info.min, info.max).astype(dtype)
    qe = np.clip(qe, info.min, info.max).astype(dtype)
    ub = ix.upper_bound(qs).astype(np.uint32).view(np.int32)
    assert np.array_equal(ub, np.searchsorted(np.sort(s), qs, side="right").astype(np.int64) - 1)
    assert np.array_equal(ix.count(qs, qe), orc.count_batch(oix, qs, qe))
    want = [bool(orc.has_overlaps(oix, a, b)) for a, b in zip(qs, qe)]
    assert np.array_equal(np.asarray(ix.has_overlaps(qs, qe)).astype(bool), want)
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nq", [786_431, 786_432, 1_000_003])
def test_count_grouped(sia, orc, dtype, nq):
    """count() on both sides of the batch size from which its queries are grouped by their ends,
    on an index of more than 4 MB, with queries around, beyond and far outside the intervals and
    inverted ones."""
    torch = pytest.importorskip("torch")
    print(f"[gpu] count grouped {np.dtype(dtype).name} nq={nq}", flush=True)
    rng = np.random.default_rng(nq)
    info = np.iinfo(dtype)
    n = 1_100_000
    s = rng.integers(-5_000_000, 60_000_000, n).astype(dtype)
    e = (s + rng.integers(0, 400, n)).astype(dtype)
    qs = rng.integers(-6_000_000, 70_000_000, nq).astype(dtype)
    qe = (qs + rng.integers(-2, 3000, nq)).astype(dtype)
    qs[:4], qe[:4] = [info.min, info.min, info.max, 7], [info.min, info.max, info.max, info.min]
    ix = _dev_index(sia, s, e)
    want = orc.count_batch(orc.build_index(s, e), qs, qe)
    c = torch.full((nq + 64,), -7, dtype=torch.int32, device="cuda")
    ix.count_device(torch.from_numpy(qs).cuda(), torch.from_numpy(qe).cuda(), c)
    torch.cuda.synchronize()
    c = c.cpu().numpy()
    assert np.array_equal(c[:nq], want) and np.all(c[nq:] == -7)
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nq", [2, 8193, 300_001])
@pytest.mark.parametrize("place", ["starts", "ends", "starts + 1"])
def test_count_over_its_queries(sia, orc, dtype, nq, place):
    """Counts written over the arrays the queries came in: a caller that needs them no more."""
    import torch
    print(f"[gpu] count over {place} {np.dtype(dtype).name} nq={nq}", flush=True)
    rng = np.random.default_rng(nq)
    n = 200_000
    s = rng.integers(0, 3_000_000, n).astype(dtype)
    e = (s + rng.integers(0, 400, n)).astype(dtype)
    qs = rng.integers(0, 3_000_000, nq).astype(dtype)
    qe = (qs + rng.integers(-2, 3000, nq)).astype(dtype)
    ix = _dev_index(sia, s, e)
    want = orc.count_batch(orc.build_index(s, e), qs, qe)
    for _ in range(3):
        tqs, tqe = torch.from_numpy(np.append(qs, [0]).astype(dtype)).cuda(), torch.from_numpy(qe).cuda()
        out = (tqe if place == "ends" else tqs).view(torch.int32)[1 if place == "starts + 1" else 0:][:nq]
        sia._native.check(sia._native.lib.siCount(ix.handle, tqs.data_ptr(), tqe.data_ptr(), nq, out.data_ptr(), None), "siCount")
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want)
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n,nq,depth", [(70_000, 1, 300), (70_000, 9, 5000), (200_000, 3000, 9000),
                                        (200_000, 40_000, 600), (100_000, 300_001, 300), (100_000, 600_001, 270)])
def test_sweep_shared_lists(sia, orc, dtype, n, nq, depth):
    """Queries whose start about `depth` intervals hold, most of them long: answered from candidate
    lists that neighbouring queries share (one list, several in turn, more candidates than one
    holds), batches that give a workgroup one query, several chunks of them, one chunk, and one
    of more than 64; queries that share with nobody, inverted ones and ones at the ends of the
    range; both orders, the values, and a capacity below the total."""
    import torch
    print(f"[gpu] sweep shared dtype={np.dtype(dtype).name} n={n} nq={nq} depth={depth}", flush=True)
    rng = np.random.default_rng(n + nq + depth)
    info = np.iinfo(dtype)
    hot = 7 * n // 5   # long intervals start below this
    s = rng.integers(0, 7 * n, n)
    long_ = rng.random(n) < 0.3
    s = np.where(long_, rng.integers(0, hot, n), s)
    e = s + np.where(long_, rng.integers(1, 2 * depth * hot // (3 * n // 10), n), rng.integers(1, 6, n))
    qs = np.where(rng.random(nq) < min(1.0, 20_000 / nq), rng.integers(0, hot, nq), rng.integers(hot, 9 * n, nq))
    qe = qs + np.where(rng.random(nq) < 0.97, rng.integers(0, 40, nq), rng.integers(-300, 60_000, nq))
    if nq > 3:
        qs[:3], qe[:3] = [info.min, info.max, info.max], [info.max, info.max, info.min]
    s, e, qs, qe = (x.astype(dtype) for x in (s, e, qs, qe))
    vals = (np.arange(n, dtype=np.int64) * 7 % 1_000_003).astype(np.int32)
    ix = _dev_index(sia, s, e, vals)
    oix = orc.build_index(s, e, vals)
    for order, mode in (("vector", 1), ("desc", 0)):
        off, idx = ix.search(qs, qe, order=order)
        ooff, oidx = orc.search_batch(oix, qs, qe, mode=mode)
        assert np.array_equal(off, ooff) and np.array_equal(idx.astype(np.int64), oidx), order
    off, v = ix.search(qs, qe, values=True)
    assert np.array_equal(v, oix["data"][oidx])
    tqs, tqe = torch.from_numpy(qs).cuda(), torch.from_numpy(qe).cuda()
    plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device="cuda")
    ix.plan_device(tqs, tqe, plan)
    toff = torch.empty(nq + 1, dtype=torch.int64, device="cuda")
    ix.offsets_planned(plan, nq, toff)
    total = int(ooff[-1])
    out = torch.full((total + 64,), -7, dtype=torch.int32, device="cuda")
    for capacity in (total - total // 3, total):
        ix.fill_planned(plan, nq, toff, out, capacity=capacity)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.array_equal(got[:capacity], oidx[:capacity]) and np.all(got[capacity:] == -7)
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nq", [1, 63, 1023, 1024, 1025, 2049, 4097, 8191, 8192, 8193, 114_687, 114_689])
def test_small_batches(sia, orc, dtype, nq):
    """Batches sorted by one workgroup, with one to eight items a thread, and the next larger forms:
    the plan is numpy's stable argsort of the ends (over the whole range, with one digit that
    varies, few distinct, all equal, and with low digits left unsorted); offsets, counts and
    lists equal the oracle's, with the counts from the plan and, planned by the learned model or
    on an index of one interval, found by the offsets pass."""
    import torch
    from superintervals_amd import autotune
    print(f"[gpu] small batches dtype={np.dtype(dtype).name} nq={nq}", flush=True)
    rng = np.random.default_rng(nq)
    info = np.iinfo(dtype)
    n = 30_000
    s = rng.integers(0, 400_000, n).astype(dtype)
    e = (s + rng.integers(0, 500, n)).astype(dtype)
    ix, one = _dev_index(sia, s, e), _dev_index(sia, s[:1], e[:1])
    model = sia.LearnedIndex(ix, 64)
    model.train(steps=20, batch=4096, lr=3e-3)
    oix, oone = orc.build_index(s, e), orc.build_index(s[:1], e[:1])
    some = rng.integers(-100, 500_000, nq)
    saved = autotune.current()
    try:
        for qe in (rng.integers(info.min, info.max, nq), 300_007 + 256 * rng.integers(0, 256, nq), rng.choice([-1, 0, 300], nq),
                   np.full(nq, 70_000), some):
            qe = qe.astype(dtype)
            qs = (qe - np.minimum(rng.integers(-20, 3000, nq), qe.astype(object) - int(info.min))).astype(dtype)
            tqs, tqe = torch.from_numpy(qs).cuda(), torch.from_numpy(qe).cuda()
            for index, o, knobs in ((ix, oix, {}), (ix, oix, {"ub_learned": 1}), (one, oone, {}),
                                    (ix, oix, {"plan_skip_low": 2, "plan_sync": 0})):
                autotune.apply(dict(saved, **knobs))
                plan = torch.full((index.plan_bytes(nq),), 0xA5, dtype=torch.uint8, device="cuda")
                index.plan_device(tqs, tqe, plan)
                off = torch.full((nq + 9,), -7, dtype=torch.int64, device="cuda")
                cnt = torch.full((nq + 8,), -7, dtype=torch.int32, device="cuda")
                index.offsets_planned(plan, nq, off, cnt)
                torch.cuda.synchronize()
                q = plan[256:256 + 4 * nq].view(torch.int32).cpu().numpy()
                low = 0xFFFF if "plan_skip_low" in knobs else 0
                assert np.array_equal(q, np.argsort(qe.astype(np.int64) & ~low, kind="stable")), knobs
                want = orc.count_batch(o, qs, qe)
                off, cnt = off.cpu().numpy(), cnt.cpu().numpy()
                assert np.array_equal(cnt[:nq], want) and np.all(cnt[nq:] == -7)
                assert np.array_equal(off[:nq + 1], np.concatenate([[0], np.cumsum(want)])) and np.all(off[nq + 1:] == -7)
            autotune.apply(saved)
        woff, widx = orc.search_batch(oix, qs, qe, mode=0)
        off, idx = ix.search(qs, qe)
        assert np.array_equal(off, woff) and np.array_equal(idx.astype(np.int64), widx)
    finally:
        autotune.apply(saved)
    model.close()
    ix.close()
    one.close()


@pytest.mark.parametrize("nq", [2, 1000, 524_287, 524_288, 524_289, 2_097_152, 2_097_153, 3_500_000])
def test_host_calls_in_chunks(sia, nq):
    """The host-buffer calls copy through pinned chunks of 2 MB, four in turn: results of one chunk,
    exactly so, one more, more than all four, from four threads at once, into buffers at odd
    places; a capacity that is too small leaves the offsets and the total."""
    import ctypes
    import threading
    print(f"[gpu] host calls in chunks nq={nq}", flush=True)
    ix = _dev_index(sia, np.array([0, 1000], np.int32), np.array([999, 2_000_000_000], np.int32), np.array([7, 9], np.int32))
    lib, bad = sia._native.lib, []

    def work(seed):
        rng = np.random.default_rng(seed)
        qs = rng.integers(0, 4000, nq).astype(np.int32)
        off, total = np.zeros(nq + 1, np.uint64), ctypes.c_uint64(0)
        want = (qs >= 1000).astype(np.uint32)
        for cap in (nq - 1, nq):
            buf = np.full(nq + 3, 77, np.uint32)
            out = buf[1:]
            rc = lib.siSearchHost(ix.handle, qs.ctypes.data, qs.ctypes.data, nq, sia.SI_ORDER_DESC, off.ctypes.data,
                                  out.ctypes.data, None, cap, ctypes.byref(total))
            ok = rc == (0 if cap == nq else sia._native.SI_ERR_CAPACITY) and total.value == nq
            ok = ok and np.array_equal(off, np.arange(nq + 1)) and buf[0] == 77 and np.all(buf[nq + 1:] == 77)
            ok = ok and (np.array_equal(out[:nq], want) if cap == nq else np.all(buf == 77))
            if not ok:
                bad.append((seed, cap, rc))
        v = np.zeros(nq, np.int32)
        rc = lib.siSearchHost(ix.handle, qs.ctypes.data, qs.ctypes.data, nq, sia.SI_ORDER_DESC, off.ctypes.data, None,
                              v.ctypes.data, nq, ctypes.byref(total))
        if rc or not np.array_equal(v, np.where(want, 9, 7)) or not np.array_equal(ix.count(qs, qs), np.ones(nq)):
            bad.append((seed, "values", rc))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4 if nq < 1_000_000 else 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("shape", ["even", "crowd", "inverted", "long", "one"])
def test_one_query_forms(sia, orc, dtype, shape):
    """Single queries, whose kernel says itself when its results are there: through the bucket tables,
    the trees (most intervals in one bucket), on an index with start > end, with a long list, of
    one interval; every mode against the oracle, ends of the range, inverted queries, no hit below
    the run and none at all, results past the scratch, and from four threads at once."""
    import threading
    print(f"[gpu] one query {np.dtype(dtype).name} {shape}", flush=True)
    rng = np.random.default_rng(5)
    info = np.iinfo(dtype)
    n = 1 if shape == "one" else 120_000
    s = rng.integers(0, 10 if shape == "crowd" else 800_000, n)
    e = s + np.where(rng.random(n) < (0.2 if shape == "long" else 0.0), rng.integers(1, 90_000, n), rng.integers(0, 9, n))
    if shape == "crowd":
        s[-1], e[-1] = 2**30, 2**30
    if shape == "inverted":
        e[::50] = s[::50] - 7
    s, e = s.astype(dtype), e.astype(dtype)
    vals = rng.integers(-5, 5, n).astype(np.int32)
    ix, oix = _dev_index(sia, s, e, vals), orc.build_index(s, e, vals)
    qs = rng.integers(-5, 800_100, 60).astype(object)
    qe = qs + rng.integers(-3, 2000, 60)
    qs = np.array(list(qs) + [info.min, info.min, info.max, 0, 2**30]).astype(dtype)
    qe = np.array(list(qe) + [info.max, info.min, info.max, 700_000, 2**30]).astype(dtype)
    bad = []

    def work(order):
        for k in order:
            a, b = qs[k:k + 1], qe[k:k + 1]
            want = orc.search(oix, qs[k], qe[k], 0)
            ok = [ix.count(a, b)[0] == want.size, bool(ix.has_overlaps(a, b)[0]) == bool(orc.has_overlaps(oix, qs[k], qe[k])),
                  np.int32(ix.upper_bound(b).view(np.int32)[0]) == np.searchsorted(np.sort(s), qe[k], side="right") - 1,
                  np.array_equal(ix.search(a, b)[1].astype(np.int64), want),
                  np.array_equal(ix.search(a, b, order="vector")[1].astype(np.int64), orc.search(oix, qs[k], qe[k], 1)),
                  np.array_equal(ix.search(a, b, values=True)[1], oix["data"][want])]
            if not all(ok):
                bad.append((int(qs[k]), int(qe[k]), ok))

    threads = [threading.Thread(target=work, args=(rng.permutation(len(qs)),)) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad[:3]
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nq", [393_215, 393_216, 1_048_575, 1_048_576, 1_100_003])
def test_grouped_forms(sia, orc, dtype, nq):
    """has_overlaps and coverage on both sides of the batch sizes from which their queries are
    grouped, on indexes that are and are not large enough for it, with queries outside the
    intervals, inverted ones, and captured in a graph (where they go ungrouped)."""
    import torch
    print(f"[gpu] grouped forms {np.dtype(dtype).name} nq={nq}", flush=True)
    rng = np.random.default_rng(nq)
    info = np.iinfo(dtype)
    for n in (65_535, 65_537, 2_100_000):
        span = 40 * n
        s = rng.integers(-1000, span, n)
        e = s + rng.integers(0, 30, n)
        qs = rng.integers(-span // 4, span + span // 4, nq)
        qe = qs + rng.integers(-2, 20, nq)
        s, e, qs, qe = (x.astype(dtype) for x in (s, e, qs, qe))
        qs[:4], qe[:4] = [info.min, info.min, info.max, 7], [info.min, info.max, info.max, info.min]
        ix, oix = _dev_index(sia, s, e), orc.build_index(s, e)
        starts = np.sort(s)
        ends = ix.download()["ends"]
        ub = np.searchsorted(starts, qe, side="right") - 1
        want = (ub >= 0) & (ends[np.maximum(ub, 0)] >= qs)
        tqs, tqe = torch.from_numpy(qs).cuda(), torch.from_numpy(qe).cuda()
        lib, check = sia._native.lib, sia._native.check
        out = torch.full((nq + 9,), 5, dtype=torch.uint8, device="cuda")
        check(lib.siHasOverlaps(ix.handle, tqs.data_ptr(), tqe.data_ptr(), nq, out.data_ptr(), None), "siHasOverlaps")
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.array_equal(got[:nq], want.astype(np.uint8)) and np.all(got[nq:] == 5)
        out.fill_(5)
        g, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.graph(g, stream=st):
            check(lib.siHasOverlaps(ix.handle, tqs.data_ptr(), tqe.data_ptr(), nq, out.data_ptr(),
                                    torch.cuda.current_stream().cuda_stream), "siHasOverlaps")
        for _ in range(2):
            g.replay()
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            assert np.array_equal(got[:nq], want.astype(np.uint8)) and np.all(got[nq:] == 5)
            out.fill_(5)
        if dtype == np.int32:
            cnt, cov = (torch.full((nq + 9,), -5, dtype=torch.int32, device="cuda") for _ in range(2))
            check(lib.siCoverage(ix.handle, tqs.data_ptr(), tqe.data_ptr(), nq, cnt.data_ptr(), cov.data_ptr(), None), "siCoverage")
            torch.cuda.synchronize()
            cnt, cov = cnt.cpu().numpy(), cov.cpu().numpy()
            assert np.array_equal(cnt[:nq], orc.count_batch(oix, qs, qe)) and np.all(cnt[nq:] == -5) and np.all(cov[nq:] == -5)
            some = np.concatenate([np.arange(200), rng.integers(0, nq, 3000), [nq - 1]])
            assert [int(cov[k]) for k in some] == [int(orc.coverage(oix, qs[k], qe[k])[1]) for k in some]
        ix.close()


@pytest.mark.parametrize("what,dtype,n,first", [
    ("count", np.int32, 1_100_000, 2_249_001), ("count", np.int64, 1_100_000, 1_124_500),
    ("count", np.int32, 25_200_000, 2_097_152), ("any", np.int32, 2_100_000, 1_835_008),
    ("coverage", np.int32, 100_000, 1_310_720), ("coverage", np.int32, 600_000, 786_432)])
def test_grouping_begins(sia, orc, what, dtype, n, first):
    """count, has_overlaps and coverage at the batch size from which queries are grouped on an index of
    n intervals, and one below it: all of the results from sorted coordinates (covered lengths of
    some queries from the oracle), queries with start > end and at the ends of the range among them,
    nothing past them written."""
    import torch
    print(f"[gpu] grouping begins {what} {np.dtype(dtype).name} n={n} nq={first}", flush=True)
    rng = np.random.default_rng(n)
    s = rng.integers(-1000, 20 * n, n)
    e = s + rng.integers(0, 60, n)
    qs = rng.integers(-5000, 20 * n + 5000, first)
    qe = qs + rng.integers(0, 90, first)
    info = np.iinfo(dtype)
    qe[:20] = qs[:20] - rng.integers(1, 90, 20)
    qs[20:24], qe[20:24] = [info.min, info.min, info.max, 7], [info.min, info.max, info.max, info.min]
    o = np.lexsort((-e, s))
    s, e = s[o].astype(dtype), e[o].astype(dtype)
    qs, qe = qs.astype(dtype), qe.astype(dtype)
    ix = sia.DeviceIndex(dtype).build(s, e, None, start_sorted=True, end_sorted=True)
    last = np.searchsorted(s, qe, side="right")
    counts = last - np.searchsorted(np.sort(e), qs)
    for k in range(24):
        counts[k] = np.count_nonzero(e[:last[k]] >= qs[k])
    any_ = (last > 0) & (e[np.maximum(last - 1, 0)] >= qs)
    oix = orc.build_index(s, e) if what == "coverage" else None
    lib, check = sia._native.lib, sia._native.check
    tqs, tqe = torch.from_numpy(qs).cuda(), torch.from_numpy(qe).cuda()
    for nq in (first - 1, first):
        out = [torch.full((first + 9,), 5, dtype=torch.uint8 if what == "any" else torch.int32, device="cuda") for _ in range(2)]
        if what == "count":
            check(lib.siCount(ix.handle, tqs.data_ptr(), tqe.data_ptr(), nq, out[0].data_ptr(), None), "siCount")
        elif what == "any":
            check(lib.siHasOverlaps(ix.handle, tqs.data_ptr(), tqe.data_ptr(), nq, out[0].data_ptr(), None), "siHasOverlaps")
        else:
            check(lib.siCoverage(ix.handle, tqs.data_ptr(), tqe.data_ptr(), nq, out[0].data_ptr(), out[1].data_ptr(), None),
                  "siCoverage")
        torch.cuda.synchronize()
        got, cov = (x.cpu().numpy() for x in out)
        assert np.array_equal(got[:nq], any_[:nq] if what == "any" else counts[:nq]) and np.all(got[nq:] == 5)
        if what == "coverage":
            assert np.all(cov[nq:] == 5)
            some = np.concatenate([np.arange(100), rng.integers(0, nq, 1000), [nq - 1]])
            assert [int(cov[k]) for k in some] == [int(orc.coverage(oix, qs[k], qe[k])[1]) for k in some]
    ix.close()


@pytest.mark.parametrize("form", ["range_skip 0", "start > end"])
@pytest.mark.parametrize("lane_steps", [1, 3, 17])
@pytest.mark.parametrize("kind", ["int32", "int64", "int64 far", "long list", "no long list"])
def test_fills_that_park_walks(sia, orc, kind, lane_steps, form):
    """Fills by the block walk (range_skip = 0, or an index that holds intervals with start > end), whose
    lanes park what exceeds lane_steps for the wave-cooperative kernel: with 32-bit ends, without
    (ends 2^40 apart), through the long list and not, in both orders and for the values.  The plan says
    that walks were parked."""
    import torch
    from superintervals_amd import autotune
    print(f"[gpu] fills that park walks {kind} lane_steps={lane_steps} {form}", flush=True)
    dtype = np.int32 if kind == "int32" else np.int64
    rng = np.random.default_rng(lane_steps)
    n, nq = 120_000, 5_000
    s = rng.integers(0, 3_000_000, n)
    long_ = rng.random(n) < 0.05
    e = s + np.where(long_, rng.integers(20_000, 400_000, n), rng.integers(0, 300, n))
    if kind == "int64 far":
        s[-50:] += np.int64(1) << 40
        e[-50:] += np.int64(1) << 40
    if form == "start > end":
        e[::400] = s[::400] - rng.integers(1, 50, n // 400)
    qs = rng.integers(-100, 3_000_000, nq)
    qe = qs + np.where(rng.random(nq) < 0.9, rng.integers(0, 2000, nq), rng.integers(-300, 80_000, nq))
    s, e, qs, qe = (x.astype(dtype) for x in (s, e, qs, qe))
    vals = rng.integers(-9, 9, n).astype(np.int32)
    saved = autotune.current()
    try:
        autotune.apply({"long_len": -1 if kind == "no long list" else 4096 if kind == "long list" else 0})
        ix = _dev_index(sia, s, e, vals)
        oix = orc.build_index(s, e, vals)
        autotune.apply(dict(saved, lane_steps=lane_steps, range_skip=int(form != "range_skip 0")))
        tqs, tqe = torch.from_numpy(qs).cuda(), torch.from_numpy(qe).cuda()
        plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device="cuda")
        off = torch.empty(nq + 1, dtype=torch.int64, device="cuda")
        ix.plan_device(tqs, tqe, plan)
        ix.offsets_planned(plan, nq, off)
        for order, mode in (("desc", 0), ("vector", 1), ("values", 0)):
            woff, widx = orc.search_batch(oix, qs, qe, mode=mode)
            assert np.array_equal(off.cpu().numpy(), woff)
            out = torch.full((int(woff[-1]) + 64,), -77, dtype=torch.int32, device="cuda")
            if order == "values":
                ix.values_fill_planned(plan, nq, off, out)
            else:
                ix.fill_planned(plan, nq, off, out, order=order)
            torch.cuda.synchronize()
            assert int(plan[4:8].view(torch.int32).item()) > 100, "no walks were parked"
            got, want = out.cpu().numpy(), oix["data"][widx] if order == "values" else widx
            assert np.array_equal(got[:len(want)], want), order
            assert np.all(got[len(want):] == -77)
    finally:
        autotune.apply(saved)
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nq", [2048 * 56, 2048 * 56 + 1])
def test_plan_sort_where_its_scan_begins(sia, dtype, nq):
    """The plan's sort on both sides of the size up to which its scatter adds the tiles' counts up itself
    (56 tiles of 2048)."""
    test_plan_sort_around_the_scan_free_size(sia, dtype, nq)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_sweep_of_full_chunks(sia, orc, dtype):
    """A batch that gives every wave of the sweep its largest chunk (256 queries), with queries that
    more than 256 intervals hold (spans of four batches in the shared lists) among queries of few
    hits: both orders and the values against the oracle."""
    print(f"[gpu] sweep of full chunks {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(3)
    n, nq = 200_000, 2_200_003
    hot = 20_000
    s = rng.integers(0, 5_000_000, n)
    s[:n // 10] = rng.integers(0, hot, n // 10)
    e = s + np.where(s < hot, rng.integers(1, 1200, n), rng.integers(0, 90, n))
    qs = rng.integers(0, 5_000_000, nq)
    qs[::1000] = rng.integers(0, hot, len(qs[::1000]))
    qe = qs + rng.integers(0, 60, nq)
    qe[7::1001] = qs[7::1001] - 30
    s, e, qs, qe = (x.astype(dtype) for x in (s, e, qs, qe))
    vals = (np.arange(n, dtype=np.int64) * 7 % 1_000_003).astype(np.int32)
    ix, oix = _dev_index(sia, s, e, vals), orc.build_index(s, e, vals)
    counts = orc.count_batch(oix, qs, qe)
    assert (counts > 300).sum() > 8_000 and counts.mean() < 6   # (the sweep's: many queries of few hits)
    for order, mode in (("desc", 0), ("vector", 1), ("values", 0)):
        off, out = ix.search(qs, qe, values=True) if order == "values" else ix.search(qs, qe, order=order)
        woff, widx = orc.search_batch(oix, qs, qe, mode=mode)
        assert np.array_equal(off, woff)
        assert np.array_equal(out, oix["data"][widx] if order == "values" else widx), order
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_fills_by_the_hits_of_the_batch(sia, orc, dtype):
    """A large batch's fill is the walk or the sweep by its hits, which only the device knows: batches
    of 2, 5 (on few intervals), 12, 20, 26 and 40 hits a query in each order say in the plan which one
    it was, and both give the oracle's lists, inverted queries and a capacity below the total included; a
    captured fill follows the hits of each replay."""
    import torch
    print(f"[gpu] fills by hits {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(8)
    nq = 1 << 20
    few = {"desc": (6, 16), "vector": (6, 22), "values": (6, 28)}
    for n, batches in ((200_000, (2, 5, 12, 20, 26, 40)), (1_500_000, (2, 12, 40))):
        span = 20 * n
        s = rng.integers(0, span, n)
        e = s + rng.integers(0, 21, n)                       # half an interval holds a point
        vals = rng.integers(-9, 9, n).astype(np.int32)
        ix, oix = _dev_index(sia, s.astype(dtype), e.astype(dtype), vals), orc.build_index(s.astype(dtype), e.astype(dtype), vals)
        dev = lambda x: torch.from_numpy(x).cuda()
        plan = torch.empty(ix.plan_bytes(nq), dtype=torch.uint8, device="cuda")
        off = torch.empty(nq + 1, dtype=torch.int64, device="cuda")
        for hits in batches:
            qs = rng.integers(0, span, nq)
            qe = qs + rng.integers(0, int(40 * (hits - 0.5)), nq)
            qe[::5003] = qs[::5003] - 7
            qs, qe = qs.astype(dtype), qe.astype(dtype)
            ix.plan_device(dev(qs), dev(qe), plan)
            ix.offsets_planned(plan, nq, off)
            for order, mode in (("desc", 0), ("vector", 1), ("values", 0)):
                woff, widx = orc.search_batch(oix, qs, qe, mode=mode)
                mean = woff[-1] / nq
                lo, hi = few[order]
                lo = lo if nq >= (n if order == "desc" else 3 * n) else 0
                want = oix["data"][widx] if order == "values" else widx
                for capacity in (int(woff[-1]), int(woff[-1]) * 2 // 3):
                    out = torch.full((len(want) + 64,), -77, dtype=torch.int32, device="cuda")
                    if order == "values":
                        sia._native.check(sia._native.lib.siSearchValuesFillPlannedBounded(
                            ix.handle, plan.data_ptr(), nq, off.data_ptr(), out.data_ptr(), capacity, None), "fill")
                    else:
                        ix.fill_planned(plan, nq, off, out, order=order, capacity=capacity)
                    torch.cuda.synchronize()
                    assert int(plan[8:12].view(torch.int32).item()) == int(not lo <= mean < hi), (n, hits, order)
                    got = out.cpu().numpy()
                    assert np.array_equal(got[:capacity], want[:capacity]) and np.all(got[capacity:] == -77), (n, hits, order)
        ix.close()
    # one captured graph, replayed for batches of either kind
    n = 300_000
    s = rng.integers(0, 20 * n, n)
    e = s + rng.integers(0, 21, n)
    s, e = s.astype(dtype), e.astype(dtype)
    ix, oix = _dev_index(sia, s, e), orc.build_index(s, e)
    tqs, tqe = torch.zeros(nq, dtype=torch.int32 if dtype == np.int32 else torch.int64, device="cuda"), None
    tqe = torch.zeros_like(tqs)
    out = torch.empty(60 * nq, dtype=torch.int32, device="cuda")
    g, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    from superintervals_amd import autotune
    saved = autotune.current()
    try:
        autotune.apply({"plan_sync": 0})
        with torch.cuda.graph(g, stream=st):
            ix.plan_device(tqs, tqe, plan, stream=st)
            ix.offsets_planned(plan, nq, off, stream=st)
            ix.fill_planned(plan, nq, off, out, capacity=out.numel(), stream=st)
        for hits, swept in ((12, 0), (40, 1), (8, 0), (3, 1), (10, 0)):
            qs = rng.integers(0, 20 * n, nq)
            qe = qs + rng.integers(0, int(40 * (hits - 0.5)), nq)
            qs, qe = qs.astype(dtype), qe.astype(dtype)
            tqs.copy_(dev(qs))
            tqe.copy_(dev(qe))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            woff, widx = orc.search_batch(oix, qs, qe, mode=0)
            assert np.array_equal(off.cpu().numpy(), woff) and np.array_equal(out[:len(widx)].cpu().numpy(), widx)
            assert int(plan[8:12].view(torch.int32).item()) == swept, hits
            _ = (out[:1000].to(torch.int64) * 3).sum().item()   # eager work between replays
    finally:
        autotune.apply(saved)
    del g
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n,keys", [(100_000, 40), (100_000, 100), (100_000, 1000), (1_200_000, 100), (1_200_000, 1000),
                                    (9_000_000, 100)])
def test_busy_buckets(sia, orc, dtype, n, keys):
    """Indexes most of whose intervals share a bucket with about `keys` others, as one interval far off
    makes them (few, busy, very busy: large counts through the plan, upper_bound and single queries
    through the trees): upper_bound, count, has_overlaps and coverage for batches below and above a
    million queries, and single queries."""
    import torch
    print(f"[gpu] busy buckets {np.dtype(dtype).name} n={n} keys={keys}", flush=True)
    rng = np.random.default_rng(n + keys)
    span = 2 * n
    s = rng.integers(0, span, n)
    s[n // 2] = min(span * keys // 4, 2**31 - 50)
    e = s + rng.integers(0, 9, n)
    o = np.lexsort((-e, s))
    s, e = s[o].astype(dtype), e[o].astype(dtype)
    ix = sia.DeviceIndex(dtype).build(s, e, None, start_sorted=True, end_sorted=True)
    by_end = np.sort(e)
    lib, check = sia._native.lib, sia._native.check
    for nq in (5000, 999_999, 1_000_001):
        qs = rng.integers(-50, span + 50, nq)
        qe = qs + rng.integers(0, 20, nq)
        qs[:3] = int(s[-1]) + np.array([-1, 0, 60])
        qe[:3] = qs[:3] + 1
        qs, qe = qs.astype(dtype), qe.astype(dtype)
        t = [torch.from_numpy(x).cuda() for x in (qs, qe)]
        out = torch.full((nq + 8,), 5, dtype=torch.int32, device="cuda")
        any_ = torch.full((nq + 8,), 5, dtype=torch.uint8, device="cuda")
        last = np.searchsorted(s, qe, side="right")
        check(lib.siUpperBound(ix.handle, t[1].data_ptr(), nq, out.data_ptr(), None), "siUpperBound")
        assert np.array_equal(out[:nq].cpu().numpy(), last - 1) and bool((out[nq:] == 5).all())
        check(lib.siCount(ix.handle, t[0].data_ptr(), t[1].data_ptr(), nq, out.data_ptr(), None), "siCount")
        counts = last - np.searchsorted(by_end, qs)
        assert np.array_equal(out[:nq].cpu().numpy(), counts) and bool((out[nq:] == 5).all())
        check(lib.siHasOverlaps(ix.handle, t[0].data_ptr(), t[1].data_ptr(), nq, any_.data_ptr(), None), "siHasOverlaps")
        assert np.array_equal(any_[:nq].cpu().numpy(), (last > 0) & (e[np.maximum(last - 1, 0)] >= qs))
        for k in range(30) if nq == 5000 else ():
            a, b = qs[k:k + 1], qe[k:k + 1]
            hits = np.flatnonzero(e[:last[k]] >= a[0])[::-1]
            assert ix.count(a, b)[0] == counts[k] and ix.upper_bound(b)[0] == np.uint32(last[k] - 1)
            assert np.array_equal(ix.search(a, b)[1].astype(np.int64), hits)
        if dtype == np.int32 and n <= 1_200_000:
            c, v = ix.coverage(qs[:2000], qe[:2000])
            oix = orc.build_index(s, e) if nq == 5000 else oix
            want = [orc.coverage(oix, a, b) for a, b in zip(qs[:300], qe[:300])]
            assert np.array_equal(c, counts[:2000]) and np.array_equal(v[:300], [w[1] for w in want])
    ix.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_busy_buckets_counted_in_a_graph(sia, dtype):
    """A large count over busy buckets takes the sorted plan, which reads back which digits vary; a
    captured one takes the tables, which need neither that nor memory: three replays over new queries,
    with eager counts between them."""
    import torch
    print(f"[gpu] busy buckets in a graph {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(8)
    n, nq, keys = 1_200_000, 1_000_001, 1000
    s = rng.integers(0, 2 * n, n)
    s[n // 2] = min(2 * n * keys // 4, 2**31 - 50)
    e = s + rng.integers(0, 9, n)
    o = np.lexsort((-e, s))
    s, e = s[o].astype(dtype), e[o].astype(dtype)
    ix = sia.DeviceIndex(dtype).build(s, e, None, start_sorted=True, end_sorted=True)
    by_end = np.sort(e)
    lib, check = sia._native.lib, sia._native.check
    t = [torch.zeros(nq, dtype=torch.int32 if dtype == np.int32 else torch.int64, device="cuda") for _ in range(2)]
    out = torch.zeros(nq, dtype=torch.int32, device="cuda")
    eager = torch.zeros(nq, dtype=torch.int32, device="cuda")
    g, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(g, stream=st):
        check(lib.siCount(ix.handle, t[0].data_ptr(), t[1].data_ptr(), nq, out.data_ptr(), st.cuda_stream), "siCount")
    for _ in range(3):
        qs = rng.integers(-50, 2 * n + 50, nq)
        qe = qs + rng.integers(0, 20, nq)
        qs, qe = qs.astype(dtype), qe.astype(dtype)
        t[0].copy_(torch.from_numpy(qs))
        t[1].copy_(torch.from_numpy(qe))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        want = np.searchsorted(s, qe, side="right") - np.searchsorted(by_end, qs)
        assert np.array_equal(out.cpu().numpy(), want)
        check(lib.siCount(ix.handle, t[0].data_ptr(), t[1].data_ptr(), nq, eager.data_ptr(), None), "siCount")
        assert np.array_equal(eager.cpu().numpy(), want)
    del g
    ix.close()


@pytest.mark.parametrize("place", ["starts", "ends"])
def test_count_in_place_in_a_graph(sia, place):
    """int32 counts written over their own queries' starts or ends, each over the word it came from: as
    without, a captured call needs no plan, whose read-back a captured stream refuses."""
    import torch
    print(f"[gpu] count in place in a graph {place}", flush=True)
    rng = np.random.default_rng(9)
    n, nq = 20_000, (1 << 22) + 77
    s = np.sort(rng.integers(0, 1_000_000, n)).astype(np.int32)
    e = s + rng.integers(0, 400, n).astype(np.int32)
    ix = sia.DeviceIndex(np.int32).build(s, e, None, start_sorted=True, end_sorted=False)
    by_end = np.sort(e)
    lib, check = sia._native.lib, sia._native.check
    t = [torch.zeros(nq, dtype=torch.int32, device="cuda") for _ in range(2)]
    out = t[0 if place == "starts" else 1]
    g, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(g, stream=st):
        check(lib.siCount(ix.handle, t[0].data_ptr(), t[1].data_ptr(), nq, out.data_ptr(), st.cuda_stream), "siCount")
    for replay in (True, True, False, True):
        qs = rng.integers(-50, 1_000_050, nq).astype(np.int32)
        qe = qs + rng.integers(0, 3000, nq).astype(np.int32)
        t[0].copy_(torch.from_numpy(qs))
        t[1].copy_(torch.from_numpy(qe))
        torch.cuda.synchronize()
        if replay:
            g.replay()
        else:
            check(lib.siCount(ix.handle, t[0].data_ptr(), t[1].data_ptr(), nq, out.data_ptr(), None), "siCount")
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), np.searchsorted(s, qe, side="right") - np.searchsorted(by_end, qs))
    del g
    ix.close()
