"""Kernels with their own edges (tiles, remainders, thresholds), bit for bit against the oracle."""
import sys
import time

import numpy as np
import pytest

from meshes import same_bits
from oracle import oracle as O
import meshoptimizer_amd as M

pytestmark = pytest.mark.gpu


def announce(what):
    print(f"[case] {what}", flush=True)
    sys.stdout.flush()


def strips(rng, sizes):
    """One mesh of disjoint triangle strips with the given vertex counts, vertices in shuffled order."""
    ibs, vs, base = [], [], 0
    for n in sizes:
        k = np.arange(n - 2)
        ibs.append(np.stack([k, k + 1 + k % 2, k + 2 - k % 2], axis=1) + base)
        x = np.arange(n) * rng.uniform(0.001, 0.01)
        p = np.stack([x, np.arange(n) % 2 * 0.05, 0.02 * rng.random(n)], axis=1) + rng.random(3) * 3
        vs.append(p.astype(np.float32))
        base += n
    order = rng.permutation(base)
    place = np.empty(base, np.int64)
    place[order] = np.arange(base)
    v = np.ascontiguousarray(np.concatenate(vs)[order])
    return place[np.concatenate(ibs)].reshape(-1).astype(np.uint32), v


@pytest.mark.parametrize("sizes", [(3, 32, 33, 34), (31, 32, 33, 4095, 4096, 4097), (8191, 8193, 3, 40), (3,) * 400 + (33,) * 70, (30011,)],
                         ids=lambda s: "-".join(map(str, s[:3])) + f"x{len(s)}")
def test_prune_component_sizes(sizes):
    """Component errors (mean and radius) around the short/long threshold and the long kernel's tile:
    with target 0 and a wide error limit every component is pruned, and the result error is the
    largest component error, bit for bit."""
    rng = np.random.default_rng(len(sizes) * 7 + sizes[0])
    ib, v = strips(rng, sizes)
    for err in (0.003, 0.05, 10.0):
        announce(f"components {sizes[:6]} x{len(sizes)} err={err}")
        rg, eg = M.simplify(ib, v, 0, err, M.SimplifyPrune | M.SimplifyLockBorder)
        ro, eo = O.simplify(ib, v, 0, err, M.SimplifyPrune | M.SimplifyLockBorder)
        assert np.array_equal(rg, ro)
        assert same_bits(eg, eo), (eg, eo)


def fan(rng, spokes, closed, soup):
    """A noisy fan of triangles around one hub in shuffled triangle order; soup: every corner its own
    vertex, so that the hub is a class of as many wedges as there are triangles."""
    ring = spokes if closed else spokes + 1
    t = np.arange(ring) * (2 * np.pi / spokes if closed else np.pi / spokes)
    p = np.stack([np.cos(t), np.sin(t), 0.1 * rng.random(ring)], axis=1) * (1 + 0.3 * rng.random((ring, 1)))
    # a second ring, so that there are edges which may collapse without the hub
    p2 = p * 1.5 + 0.01 * rng.random((ring, 3))
    v = np.concatenate([[[0, 0, 0.2]], p, p2]).astype(np.float32)
    k = np.arange(spokes)
    a, b = 1 + k, 1 + (k + 1) % ring
    tri = np.concatenate([np.stack([np.zeros_like(a), a, b], 1), np.stack([a, a + ring, b], 1), np.stack([b, a + ring, b + ring], 1)])
    tri = tri[rng.permutation(len(tri))]
    if soup:
        return np.arange(3 * len(tri), dtype=np.uint32), np.ascontiguousarray(v[tri.reshape(-1)])
    return tri.reshape(-1).astype(np.uint32), v


@pytest.mark.parametrize("soup", [False, True])
@pytest.mark.parametrize("spokes", [6, 7, 8, 9, 63, 64, 65, 66, 129, 700])
def test_vertex_valence(spokes, soup):
    """Corner lists around the sorting network's eight, the wavefront's 64 and beyond, open edges, and
    adjacency lists around the length that goes to a whole wavefront."""
    rng = np.random.default_rng(spokes)
    for closed in (True, False):
        ib, v = fan(rng, spokes, closed, soup)
        for opts in (0, M.SimplifyLockBorder, M.SimplifyPermissive):
            announce(f"fan {spokes} closed={closed} soup={soup} opts={opts}")
            for target in (ib.size // 6 * 3, 0):
                rg, eg = M.simplify(ib, v, target, 0.5, opts)
                ro, eo = O.simplify(ib, v, target, 0.5, opts)
                assert np.array_equal(rg, ro)
                assert same_bits(eg, eo), (eg, eo)


def padded(rng, side, padding):
    """A grid with (0,0,0) triangles between its own, as padded index buffers hold them."""
    from meshoptimizer_amd import workloads as W
    m = W.grid(side, seed=padding)
    tri = np.concatenate([m.indices.reshape(-1, 3), np.zeros((padding, 3), np.uint32)])
    return tri[rng.permutation(len(tri))].reshape(-1).astype(np.uint32), m.vertices[:, :3].copy()


def long_list_case(name, rng):
    kind, size = name.rstrip("0123456789"), int("".join(c for c in name if c.isdigit()))
    if kind == "padding":
        return padded(rng, 24, size)
    if kind == "fan":
        return fan(rng, size, bool(size & 1), False)
    if kind == "soupfan":
        return fan(rng, size, bool(size & 1), True)
    if kind == "point":
        # `size` vertices at one position, each in a triangle with two vertices of a grid
        ib, v = padded(rng, 30, 0)
        n = v.shape[0]
        own = np.arange(n, n + size)
        tri = np.stack([own, rng.integers(0, n, size), rng.integers(0, n, size)], axis=1)
        tri = np.concatenate([ib.reshape(-1, 3), tri])
        v = np.concatenate([v, np.full((size, 3), 0.37, np.float32)]).astype(np.float32)
        return tri[rng.permutation(len(tri))].reshape(-1).astype(np.uint32), v
    if kind == "snapped":
        # few positions of many vertices, the primaries neighbours in index order
        v = (np.floor(rng.random((size, 3)) * 4) / 4).astype(np.float32)
        return rng.integers(0, size, size * 9).astype(np.uint32), v
    if kind == "strips":
        # vertices of about 20 corners, all in one wavefront's lists or not
        return (rng.integers(0, size, (size * 20 // 3, 3)).reshape(-1).astype(np.uint32), rng.random((size, 3)).astype(np.float32))
    if kind == "crowd":
        # the lists of one wavefront, each of more than `size` corners
        ib = np.concatenate([np.repeat(np.arange(64), size), rng.integers(0, 64, 64 * size * 2)]).astype(np.uint32)
        return np.ascontiguousarray(ib.reshape(3, -1).T).reshape(-1), rng.random((64, 3)).astype(np.float32)
    # every list long, with edges repeated and self edges
    return rng.integers(0, 37, (size, 3)).reshape(-1).astype(np.uint32), rng.random((37, 3)).astype(np.float32)


@pytest.mark.parametrize("name", ["padding84", "padding95", "padding96", "padding7000", "fan255", "fan257", "fan285", "fan288", "fan513", "fan4000", "fan4001",
                                  "soupfan255", "soupfan257", "soupfan285", "soupfan288", "soupfan513", "soupfan3000", "soupfan3001", "point255",
                                  "point285", "point287", "point513", "point6000", "dense3100", "dense20000", "snapped300", "snapped1000",
                                  "snapped4000", "strips40", "strips64", "strips70", "strips500"])
def test_long_corner_lists(name):
    """Corner lists and open edges around the work from which lists are sorted and edges come from a
    table, in one list and in many of one wavefront, by vertex and by class, in every option that
    reads them."""
    rng = np.random.default_rng(len(name) + int("".join(c for c in name if c.isdigit())))
    ib, v = long_list_case(name, rng)
    a, w = rng.random((v.shape[0], 2)).astype(np.float32), np.array([0.3, 0.1], np.float32)
    for opts, attrs in ((0, False), (M.SimplifyLockBorder, True), (M.SimplifyPermissive, False), (M.SimplifySparse | M.SimplifyPrune, True)):
        announce(f"long lists {name} opts={opts} attributes={attrs}")
        target = ib.size // 12 * 3
        rg, eg = M.simplify_with_attributes(ib, v, a if attrs else None, w if attrs else None, None, target, 0.3, opts)
        call, _ = M.last_call_stats()
        ro, eo, st = O.simplify(ib, v, target, 0.3, opts, attributes=a if attrs else None, weights=w if attrs else None, stats=True)
        assert call["kinds"] == list(st.kinds)
        assert np.array_equal(rg, ro)
        assert same_bits(eg, eo), (eg, eo)


@pytest.mark.parametrize("name", ["padding100000", "point100000", "crowd22000"])
def test_long_corner_lists_time(name):
    """A list of a hundred thousand corners or more, and 64 such lists, cost time linear in them (their
    pairs would take many seconds)."""
    ib, v = long_list_case(name, np.random.default_rng(5))
    assert name[:5] != "crowd" or np.bincount(ib).min() >= 65536
    M.simplify(ib, v, ib.size // 12 * 3, 1e-3, 0)
    announce(f"long lists {name}")
    t = time.perf_counter()
    M.simplify(ib, v, ib.size // 12 * 3, 1e-3, 0)
    assert time.perf_counter() - t < 1.0


@pytest.mark.parametrize("attributes", [1, 3, 4, 5, 8, 9])
def test_attribute_counts(attributes):
    """Gradients in groups of four: below, at and above a group."""
    from meshoptimizer_amd import workloads as W
    rng = np.random.default_rng(attributes)
    m = W.grid(41, seed=attributes)
    a = rng.random((m.vertex_count, attributes)).astype(np.float32) * np.float32(0.2)
    w = (0.1 + rng.random(attributes)).astype(np.float32)
    announce(f"attributes {attributes}")
    target = W.target_count(m.index_count, 1, 5)
    rg, eg = M.simplify_with_attributes(m.indices, m.vertices, a, w, None, target, 0.1, 0)
    ro, eo = O.simplify(m.indices, m.vertices, target, 0.1, 0, attributes=a, weights=w)
    assert np.array_equal(rg, ro)
    assert same_bits(eg, eo), (eg, eo)


@pytest.mark.parametrize("side", [2, 3, 16, 17, 24, 25, 105, 106, 147, 209])
def test_candidate_tiles(side):
    """Triangle and candidate counts around the tiles of the compaction and of the one-pass sort (1024
    and 2048 candidates a tile: grids of about 3 n^2 candidates), down to one cell."""
    from meshoptimizer_amd import workloads as W
    m = W.grid(side, seed=side)
    for num, den, err in ((0, 1, 1.0), (1, 2, 1e-2)):
        target = W.target_count(m.index_count, num, den)
        announce(f"grid {side} target {target} err {err}")
        rg, eg = M.simplify(m.indices, m.vertices, target, err, 0)
        ro, eo = O.simplify(m.indices, m.vertices, target, err, 0)
        assert np.array_equal(rg, ro)
        assert same_bits(eg, eo), (eg, eo)


@pytest.mark.parametrize("mesh", ["grid3", "grid20", "grid110", "grid220", "grid330", "fan8", "fan9", "fan17", "fan200"])
def test_deep_rounds(mesh):
    """Rounds that examine moving corners from the first on: lists that leave a wavefront 8, 16, 32 and
    64 ranks, and sources of more triangles than the lanes that test them."""
    from meshoptimizer_amd import workloads as W
    size = int("".join(c for c in mesh if c.isdigit()))
    if mesh.startswith("grid"):
        m = W.grid(size, seed=size)
        ib, v = m.indices, m.vertices
    else:
        ib, v = fan(np.random.default_rng(size), size, True, False)
    M.set_round_policy(-1, 0)
    try:
        for den, err, opts in ((10, 1.0, 0), (2, 1e-2, M.SimplifyPermissive)):
            target = W.target_count(ib.size, 1, den)
            announce(f"deep {mesh} target 1/{den} err {err}")
            rg, eg = M.simplify(ib, v, target, err, opts)
            ro, eo = O.simplify(ib, v, target, err, opts)
            assert np.array_equal(rg, ro)
            assert same_bits(eg, eo), (eg, eo)
    finally:
        M.set_round_policy()


@pytest.mark.parametrize("side,grid", [(2, 2), (17, 3), (27, 3), (27, 26), (64, 4), (64, 20), (300, 6), (300, 150), (516, 40)])
def test_sloppy_cells(side, grid):
    """Cells of few and of many triangles (both forms of the cell sums) and entry counts around the
    sort's tile, with runs of vertices in one cell longer and shorter than a wavefront; locked
    vertices are cells of their own."""
    rng = np.random.default_rng(side * 1000 + grid)
    g = np.linspace(0, 1, side, dtype=np.float32)
    x, y = np.meshgrid(g, g)
    v = np.stack([x.ravel(), y.ravel(), 0.1 * rng.random(side * side).astype(np.float32)], axis=1).astype(np.float32)
    q = (np.arange(side - 1)[:, None] * side + np.arange(side - 1)).ravel()
    ib = np.stack([q, q + 1, q + side, q + 1, q + side + 1, q + side], axis=1).reshape(-1).astype(np.uint32)
    for lock in (None, (rng.random(side * side) < 0.02).astype(np.uint8)):
        for target in (0, ib.size // 3 // 4 * 3):
            announce(f"sloppy cells side={side} grid={grid} lock={lock is not None} target={target}")
            rg, eg = M.simplify_sloppy(ib, v, target, 1.0 / grid, lock=lock)
            ro, eo = O.simplify_sloppy(ib, v, target, 1.0 / grid, lock=lock)
            assert np.array_equal(rg, ro)
            assert same_bits(eg, eo), (eg, eo)
