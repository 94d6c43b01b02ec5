"""GPU tests of the serving loop (meshopt_hip_server_*): each request's result in a concurrent
mix equals the same request run alone (meshopt_simplify / meshopt_simplifyWithAttributes) and the
oracle, bit for bit; admission honours the memory budget; invalid requests are rejected."""
import sys

import numpy as np
import pytest

from meshes import random_grid, random_soup, same_bits
from oracle import oracle as O
import meshoptimizer_amd as M
from meshoptimizer_amd import workloads as W

pytestmark = pytest.mark.gpu


def announce(what):
    print(f"[case] {what}", flush=True)
    sys.stdout.flush()


def mixed_requests(seed=3):
    """Requests of very different sizes and kinds: grids, icospheres, seamed grids with
    attributes, random soups with vertex locks."""
    rng = np.random.default_rng(seed)
    out = []
    for k in range(14):
        kind = k % 5
        if kind == 0:
            m = W.grid(int(rng.integers(20, 160)), seed=int(rng.integers(1, 1000)))
            out.append(dict(ib=m.indices, v=m.vertices, target=W.target_count(m.index_count, 1, 4), err=1e-2, opts=0))
        elif kind == 1:
            m = W.icosphere(int(rng.integers(2, 7)), seed=int(rng.integers(1, 1000)))
            out.append(dict(ib=m.indices, v=m.vertices, target=W.target_count(m.index_count, 1, 10), err=1e-2, opts=0))
        elif kind == 2:
            m = W.seamed_grid(int(rng.integers(16, 96)), seams=2, seed=int(rng.integers(1, 1000)))
            out.append(dict(ib=m.indices, v=m.vertices, target=W.target_count(m.index_count, 1, 5), err=1e-2, opts=0,
                            attrs=m.vertices[:, 3:8], weights=W.SEAMED_GRID_WEIGHTS))
        elif kind == 3:
            ib, v = random_soup(rng, nv=int(rng.integers(50, 400)), ntri=int(rng.integers(50, 800)))
            lock = rng.integers(0, 8, size=v.shape[0]).astype(np.uint8)
            out.append(dict(ib=ib, v=v, target=ib.size // 2 // 3 * 3, err=1e-1, opts=M.SimplifyPermissive,
                            attrs=v[:, 3:4], weights=np.array([0.5], np.float32), lock=lock))
        else:
            ib, v = random_grid(rng, n=int(rng.integers(6, 30)))
            out.append(dict(ib=ib, v=v, target=0, err=float(rng.choice([1e-3, 1e-2, 1e-1])),
                            opts=int(rng.choice([0, M.SimplifyLockBorder, M.SimplifyRegularize, M.SimplifyErrorAbsolute]))))
    return out


def alone(r):
    if "attrs" in r or "lock" in r:
        return M.simplify_with_attributes(r["ib"], r["v"], r.get("attrs"), r.get("weights"), r.get("lock"), r["target"],
                                          r["err"], r["opts"])
    return M.simplify(r["ib"], r["v"], r["target"], r["err"], r["opts"])


def submit(srv, r):
    return srv.submit(r["ib"], r["v"], r["target"], r["err"], r["opts"], attributes=r.get("attrs"), weights=r.get("weights"),
                      lock=r.get("lock"))


@pytest.mark.parametrize("V,T,A,opts,budget", [
    (4, 2, 0, 0, 25696), (4, 2, 3, 8, 27296), (100, 200, 0, 0, 130976), (1000, 20, 0, 0, 280736), (1000, 20, 0, 2, 69216),
    (1000, 20, 3, 8, 441376), (1000, 2000, 0, 0, 1136416), (1000, 2000, 3, 2, 1382176), (11000, 22000, 0, 8, 12508256),
    (100000, 3000, 0, 0, 26785696), (100000, 3000, 0, 2, 5656096), (30000, 58000, 3, 0, 37294496), (120000, 174900, 0, 0, 106311456),
    (300000, 620000, 0, 8, 350150496), (400000, 800000, 0, 0, 449525216), (1500000, 100, 3, 8, 623377696)])
def test_budgets_that_were_enough(V, T, A, opts, budget):
    """Requests of many vertices, many triangles, attributes, Sparse and Prune, each with the budget that
    a single adjacency and separate set-up arrays needed: they are still admitted, and run."""
    rng = np.random.default_rng(V + T)
    ib = rng.integers(0, V, 3 * T).astype(np.uint32)
    v = rng.random((V, 3 + A)).astype(np.float32)
    announce(f"budget V={V} T={T} A={A} opts={opts}")
    with M.Server(budget_bytes=budget, slots=1) as srv:
        ri, _, info = srv.wait(srv.submit(ib, v, ib.size, 1e-2, opts, attributes=v[:, 3:] if A else None,
                                          weights=np.ones(A, np.float32) if A else None))
    assert info["device_bytes"] <= budget
    assert np.array_equal(ri, ib)


def test_mix_equals_alone_and_oracle():
    reqs = mixed_requests()
    announce(f"serving mix of {len(reqs)} requests on 4 slots")
    with M.Server(budget_bytes=8 << 30, slots=4) as srv:
        tickets = [submit(srv, r) for r in reqs]
        results = [srv.wait(t) for t in tickets]
    for k, (r, (ri, re, info)) in enumerate(zip(reqs, results)):
        ai, ae = alone(r)
        assert np.array_equal(ri, ai) and same_bits(re, ae), f"request {k}: mix differs from the request alone"
        oi, oe = O.simplify(r["ib"], r["v"], r["target"], r["err"], r["opts"], attributes=r.get("attrs"),
                            weights=r.get("weights"), lock=r.get("lock"))
        assert np.array_equal(ri, oi) and same_bits(re, oe), f"request {k}: differs from the oracle"
    # the slots ran side by side: some request started before another one on a different slot finished
    spans = [(i["start_ms"], i["finish_ms"], i["slot"]) for _, _, i in results]
    overlap = any(a[0] < b[1] and b[0] < a[1] and a[2] != b[2] for x, a in enumerate(spans) for b in spans[x + 1:])
    assert overlap, "no two requests overlapped in time"
    assert len({s for _, _, s in spans}) > 1


def test_budget_serialises_admission():
    m = W.icosphere(5, seed=7)
    target = W.target_count(m.index_count, 1, 4)
    announce("budget admission")
    with M.Server(budget_bytes=8 << 30, slots=1) as srv:
        _, _, info = srv.wait(srv.submit(m.indices, m.vertices, target))
    need = info["device_bytes"]
    expect = M.simplify(m.indices, m.vertices, target)
    # room for one request at a time: three slots, but the requests must run one after another
    with M.Server(budget_bytes=need * 3 // 2, slots=3) as srv:
        tickets = [srv.submit(m.indices, m.vertices, target) for _ in range(3)]
        results = [srv.wait(t) for t in tickets]
    for ri, re, _ in results:
        assert np.array_equal(ri, expect[0]) and same_bits(re, expect[1])
    spans = sorted((i["start_ms"], i["finish_ms"]) for _, _, i in results)
    for a, b in zip(spans, spans[1:]):
        assert b[0] >= a[1], f"requests overlapped under a budget that fits one: {spans}"


def test_rejections():
    announce("rejections")
    m = W.grid(64)
    with M.Server(budget_bytes=1 << 20, slots=2) as srv:
        with pytest.raises(RuntimeError, match="budget"):
            srv.submit(m.indices, m.vertices, 0)
    with M.Server(budget_bytes=1 << 30, slots=2) as srv:
        with pytest.raises(RuntimeError, match="invalid"):
            srv.submit(m.indices, m.vertices, m.index_count + 3)
        bad = m.indices.copy()
        bad[5] = m.vertex_count + 10
        t_bad = srv.submit(bad, m.vertices, 0)
        t_ok = srv.submit(m.indices, m.vertices, W.target_count(m.index_count, 1, 4))
        with pytest.raises(RuntimeError, match="vertex"):
            srv.wait(t_bad)
        ri, re, _ = srv.wait(t_ok)
    e = M.simplify(m.indices, m.vertices, W.target_count(m.index_count, 1, 4))
    assert np.array_equal(ri, e[0]) and same_bits(re, e[1])


def test_small_requests_batched():
    """Small requests queued together run as one batched call on their slot, and each result still
    equals the oracle.  A large request submitted first keeps the one slot busy while the small
    ones queue behind it.  A batch takes the compatible requests from anywhere in the queue: the
    request with other options and the runs with locks or attributes in between do not stop the
    last four plain requests from joining the first batch.  Requests with attributes (one weight
    set) batch together; a run with locks batches too; and the run holding a request with a bad
    index falls back to one call per request, failing only that one."""
    rng = np.random.default_rng(77)
    big = W.icosphere(8, seed=5)
    reqs = [dict(ib=big.indices, v=big.vertices, target=W.target_count(big.index_count, 1, 10), err=1e-2, opts=0)]
    for k in range(64):
        if 50 <= k < 60:
            m = W.seamed_grid(int(rng.integers(6, 20)), seams=2, seed=int(rng.integers(1, 1000)))
            ib, v = m.indices, m.vertices
        else:
            ib, v = random_grid(rng, n=int(rng.integers(4, 24)))
        r = dict(ib=ib, v=v, target=(ib.size // 3 * int(rng.integers(1, 4)) // 4) * 3, err=1e-2, opts=M.SimplifyLockBorder)
        if k == 24:
            r.update(err=1e-1, opts=0)
        if 25 <= k < 50:
            r["lock"] = (rng.integers(0, 8, size=v.shape[0]) * (rng.random(v.shape[0]) < 0.3)).astype(np.uint8)
        if 50 <= k < 60:
            r.update(attrs=v[:, 3:8], weights=W.SEAMED_GRID_WEIGHTS)
        reqs.append(r)
    bad_at = 1 + 40
    bad = reqs[bad_at]["ib"].copy()
    bad[4] = reqs[bad_at]["v"].shape[0] + 3
    announce(f"serving: {len(reqs)} requests on one slot, small ones batched, a bad index at {bad_at}")

    with M.Server(budget_bytes=8 << 30, slots=1) as srv:
        tickets = [srv.submit(bad if k == bad_at else r["ib"], r["v"], r["target"], r["err"], r["opts"], attributes=r.get("attrs"),
                              weights=r.get("weights"), lock=r.get("lock")) for k, r in enumerate(reqs)]
        results = []
        for k, t in enumerate(tickets):
            if k == bad_at:
                with pytest.raises(RuntimeError, match="vertex"):
                    srv.wait(t)
                results.append(None)
            else:
                results.append(srv.wait(t))
    for k, (r, res) in enumerate(zip(reqs, results)):
        if res is None:
            continue
        ri, re, info = res
        oi, oe = O.simplify(r["ib"], r["v"], r["target"], r["err"], r["opts"], attributes=r.get("attrs"), weights=r.get("weights"),
                            lock=r.get("lock"))
        assert np.array_equal(ri, oi) and same_bits(re, oe), f"request {k}: differs from the oracle (batched {info['batched']})"
    info = [None if res is None else res[2] for res in results]
    assert info[0]["batched"] == 1, "the large request runs on the plain path"
    first = [k for k in range(1, len(reqs)) if info[k] is not None and info[k]["start_ms"] == info[1]["start_ms"]]
    assert first == list(range(1, 25)) + list(range(61, 65)), f"the first batch took {first}"
    assert all(info[k]["batched"] == 28 for k in first)
    assert info[25]["batched"] == 1, "the request with other options runs alone"
    assert all(info[k]["batched"] == 10 for k in range(51, 61)), "the requests with attributes run as one batch"
    # a group shares its start time; the one holding the bad index ran request by request
    locked = [info[k] for k in range(26, 51) if k != bad_at]
    assert len({i["start_ms"] for i in locked}) == 1 and all(i["batched"] == 1 for i in locked), \
        "the run with a bad index did not fall back to one call per request"


def test_batches_split_by_attribute_weights():
    """Requests with attributes batch only with requests of the same attribute count and weights:
    32 seamed grids queued behind a large request on one slot, with 3 or 5 attributes and one of
    two weight sets each, run as four batches, one per (count, weights), and every result equals
    the oracle."""
    rng = np.random.default_rng(91)
    big = W.icosphere(8, seed=9)
    reqs = [dict(ib=big.indices, v=big.vertices, target=W.target_count(big.index_count, 1, 10), err=1e-2, opts=0)]
    w5 = [W.SEAMED_GRID_WEIGHTS, np.array([0.25, 0.5, 1.0, 2.0, 0.125], np.float32)]
    keys = []
    for k in range(32):
        m = W.seamed_grid(int(rng.integers(6, 20)), seams=2, seed=int(rng.integers(1, 1000)))
        count, which = (3, 5)[k % 2], (k // 2) % 2
        weights = w5[which][:count].copy()
        reqs.append(dict(ib=m.indices, v=m.vertices, target=(m.index_count // 3 * int(rng.integers(1, 4)) // 4) * 3, err=1e-2,
                         opts=M.SimplifyLockBorder, attrs=m.vertices[:, 3:3 + count], weights=weights))
        keys.append((count, which))
    announce(f"serving: {len(reqs)} requests, attribute batches split by count and weights")
    with M.Server(budget_bytes=8 << 30, slots=1) as srv:
        tickets = [srv.submit(r["ib"], r["v"], r["target"], r["err"], r["opts"], attributes=r["attrs"] if "attrs" in r else None,
                              weights=r.get("weights")) for r in reqs]
        results = [srv.wait(t) for t in tickets]
    for k, (r, (ri, re, info)) in enumerate(zip(reqs, results)):
        oi, oe = O.simplify(r["ib"], r["v"], r["target"], r["err"], r["opts"], attributes=r.get("attrs"), weights=r.get("weights"))
        assert np.array_equal(ri, oi) and same_bits(re, oe), f"request {k}: differs from the oracle (batched {info['batched']})"
    assert results[0][2]["batched"] == 1
    from collections import Counter
    sizes = Counter(keys)
    for k, key in enumerate(keys):
        assert results[k + 1][2]["batched"] == sizes[key], f"request {k + 1}: batched {results[k + 1][2]['batched']}, expected {sizes[key]}"
    starts = {key: {results[k + 1][2]["start_ms"] for k, kk in enumerate(keys) if kk == key} for key in sizes}
    assert all(len(v) == 1 for v in starts.values()), f"a (count, weights) group ran in more than one call: {starts}"
