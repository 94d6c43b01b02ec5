"""Kernels with their own edges (tiles, remainders, thresholds), bit for bit against the oracle."""
import sys

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
