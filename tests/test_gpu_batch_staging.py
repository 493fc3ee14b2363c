"""Plane batches at the edges of their staging: in pinned memory (up to 1024 entries), in the context's
device array (up to 65536), in an allocation of their own; larger after smaller and smaller after
larger, and from several threads of one context. A batch's entries do not depend on each other, so
every size holds the same bits as one entry at a time does, and the same as the staging without
allocation where that takes it.
"""
import threading

import numpy as np
import pytest

from ns_multiphase_amd import workloads as W

pytestmark = pytest.mark.gpu


def _entries(m):
    rng = np.random.default_rng(m)
    n = rng.standard_normal((m, 3))
    n /= np.sqrt((n ** 2).sum(1))[:, None]
    return rng.integers(1, 17, (m, 3)), n, rng.random(m)


def test_batches_of_every_staging_hold_the_same_bits():
    from ns_multiphase_amd import solver
    ctx = solver.Context(W.deformation3d(16)[0])
    ijk, n, vf = _entries(65540)
    want = np.concatenate([ctx.plic_dist_batch_noalloc(ijk[q], n[q], vf[q])
                           for q in (slice(0, 65536), slice(65536, None))])
    for m in (1, 1024, 1025, 65536, 65537, 65540, 1025, 63):
        d = ctx.plic_dist_batch(ijk[:m], n[:m], vf[:m])
        assert np.array_equal(d, want[:m])
    back = ctx.plic_vf_batch(ijk, n, want)
    assert np.abs(back - vf).max() <= 1e-12
    for m in (1, 64, 1024, 1025, 65536):
        assert np.array_equal(ctx.plic_vf_batch(ijk[-m:], n[-m:], want[-m:]), back[-m:])


def test_batches_from_threads():
    from ns_multiphase_amd import solver
    ctx = solver.Context(W.deformation3d(16)[0])
    sets = [_entries(m) for m in (64, 700, 3000, 1024)]
    want = [ctx.plic_dist_batch_noalloc(*s) for s in sets]
    bad = []

    def run(q):
        for _ in range(20):
            if not np.array_equal(ctx.plic_dist_batch(*sets[q]), want[q]):
                bad.append(q)

    threads = [threading.Thread(target=run, args=(q,)) for q in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_large_batches_from_threads():
    """Batches with allocations of their own, beside each other and beside staged ones."""
    from ns_multiphase_amd import solver
    ctx = solver.Context(W.deformation3d(16)[0])
    sets = [_entries(m) for m in (65537, 70001, 65536, 1000)]
    want = [np.concatenate([ctx.plic_dist_batch_noalloc(*(a[q:q + 65536] for a in s)) for q in range(0, len(s[2]), 65536)])
            for s in sets]
    bad = []

    def run(q):
        for _ in range(8):
            if not np.array_equal(ctx.plic_dist_batch(*sets[q]), want[q]):
                bad.append(q)

    threads = [threading.Thread(target=run, args=(q,)) for q in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
