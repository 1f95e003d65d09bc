"""Neighbour lists whose arrays hold exactly the pairs: every chunk that a wave leaves partly empty lies
below the pair count or in the spill, and the list comes out dense and whole."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def keys(i, j):
    import torch
    return torch.sort(torch.minimum(i, j).long() << 32 | torch.maximum(i, j).long())[0]


# pairs: 5e3 (chunks of 64 slots), 1.3e6, 2e7 (512), 6e7 (2048, spill of 512 each)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,side,clumps", [(700, 6.0, 0), (40_000, 17.0, 0), (100_000, 10.0, 0), (100_000, 7.0, 0),
                                           (60_000, 12.0, 6)])
def test_list_without_a_slot_to_spare(clm, n, side, clumps, dtype):
    import torch
    print(f"[capacity] n={n} side={side} clumps={clumps} {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.random((n, 3)) * side
    if clumps:
        x = (x[rng.integers(0, clumps, n)] + rng.normal(0, 0.5, (n, 3))) % side
    xt = torch.as_tensor(x.astype(dtype)).cuda()
    s = clm.ParticleSystem(xpositions=xt, unitcell=[side] * 3, cutoff=1.0)
    counts = clm.pairwise_(clm.DistanceHistogram(1, 1.0), s)
    pairs = int(counts.sum())
    s = clm.ParticleSystem(xpositions=xt, unitcell=[side] * 3, cutoff=1.0)
    roomy = clm.pairwise_(clm.NeighborListOp(capacity=pairs + pairs // 3 + 100), s, device_output=True)
    assert len(roomy) == pairs
    want = keys(roomy.i, roomy.j)
    i, j = (torch.full((pairs,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    d = torch.empty(pairs, dtype=xt.dtype, device="cuda")
    m = C.c_int64()
    torch.cuda.synchronize()
    p = lambda t: C.c_void_p(t.data_ptr())
    s._ctx.check(s._ctx.lib.clm_neighborlist(s._ctx.ptr, p(i), p(j), p(d), pairs, C.byref(m), 1), "list")
    assert m.value == pairs and torch.equal(keys(i, j), want)
