"""Contexts made and destroyed one after another and side by side: what a destroyed one leaves
for the next (memory, a stream, a read-back block) is bounded and carries nothing over."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = [(1, 3, np.float64, None), (300, 2, np.float32, 1.0), (4_001, 3, np.float32, None), (30_000, 3, np.float64, 1.0)]


def one(clm, k):
    n, dim, dtype, side = KINDS[k]
    x = np.random.default_rng(k).random((n, dim)).astype(dtype)
    r = clm.neighborlist(xpositions=x, unitcell=None if side is None else np.full(dim, side), cutoff=0.07, lcell=1 + k % 2)
    o = np.lexsort((r.d, np.maximum(r.i, r.j), np.minimum(r.i, r.j)))
    return np.minimum(r.i, r.j)[o], np.maximum(r.i, r.j)[o], r.d[o]


def same(a, b):
    return all(np.array_equal(u, v) for u, v in zip(a, b))


@pytest.mark.parametrize("threads", [1, 4])
def test_contexts_in_turn_and_side_by_side(clm, O, threads):
    want = []
    for k, (n, dim, dtype, side) in enumerate(KINDS):
        x = np.random.default_rng(k).random((n, dim)).astype(dtype)
        if side is None:
            box = O.make_nonperiodic_box(x, 0.07, lcell=1 + k % 2, dtype=dtype)
        else:
            box = O.make_box(np.full(dim, side), 0.07, lcell=1 + k % 2, dtype=dtype)
        i, j, _, d = O.pairs(box, x, 1)
        lo, hi = np.minimum(i, j), np.maximum(i, j)
        o = np.lexsort((d, hi, lo))
        want.append((lo[o], hi[o], d[o].astype(dtype)))
    wrong = []

    def work(t):
        for r in range(6):
            k = (t + r) % len(KINDS)
            if not same(one(clm, k), want[k]):
                wrong.append((t, r, k))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong


def test_what_contexts_leave_is_bounded(clm):
    import torch
    x = np.random.default_rng(0).random((400_000, 3))
    free = []
    for r in range(12):
        s = clm.ParticleSystem(xpositions=x[: 30_000 * (1 + r)], unitcell=[1.0] * 3, cutoff=0.04)
        clm.pairwise_(clm.NeighborListOp(), s)
        s._ctx.close()
        free.append(torch.cuda.mem_get_info()[0])
    assert free[0] - min(free) <= (256 << 20) + (64 << 20)


def test_a_system_ends_with_its_last_reference(clm):
    """No cycle keeps a system (and its device memory) alive after its list is taken, and a list
    that a later one overwrote is still refused when the system is gone."""
    import gc
    import weakref
    x = np.random.default_rng(1).random((500, 3))
    gc.disable()
    try:
        s = clm.ParticleSystem(xpositions=x, unitcell=[1.0] * 3, cutoff=0.2)
        first = clm.pairwise_(clm.NeighborListOp(), s)
        last = clm.pairwise_(clm.NeighborListOp(), s)
        n, gone = len(last), weakref.ref(s)
        del s
        assert gone() is None
    finally:
        gc.enable()
    assert len(last.i) == n
    with pytest.raises(clm.StaleResultError):
        first.i
