"""Grids of cells on both sides of the line above which the homes of cells are counted and scanned
apart, nearly empty ones and one of cells in parts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "open"])
@pytest.mark.parametrize("dim,side,lcell", [(3, 63.0, 1), (3, 64.0, 1), (3, 65.0, 1), (3, 65.0, 3), (2, 544.5, 1), (2, 545.5, 1)])
def test_sparse_grids(clm, O, dim, side, lcell, kind, dtype):
    n = 4000
    print(f"[grids] dim={dim} side={side} lcell={lcell} {kind} {np.dtype(dtype).name}", flush=True)
    x = np.random.default_rng(dim).random((n, dim)) * (side if lcell == 1 else 1.2 * side / 3)
    x[:600] *= 0.05  # (and some pairs)
    x = x.astype(dtype)
    uc = None if kind == "open" else np.full(dim, side if lcell == 1 else 1.2 * side / 3)
    box = O.make_nonperiodic_box(x, 1.0, lcell=lcell, dtype=dtype) if uc is None else O.make_box(uc, 1.0, lcell=lcell, dtype=dtype)
    i, j, _, do = O.pairs(box, x, 1)
    lo, hi = np.minimum(i, j), np.maximum(i, j)
    o = np.lexsort((do, hi, lo))
    s = clm.ParticleSystem(xpositions=x, unitcell=uc, cutoff=1.0, lcell=lcell)
    for _ in range(2):
        a, b, d = clm.pairwise_(clm.NeighborListOp(), s).canonical()
        k = np.lexsort((d, b, a))
        assert len(d) and np.array_equal(a[k], lo[o]) and np.array_equal(b[k], hi[o])
        assert np.array_equal(d[k].astype(np.float64), do[o])
        clm.update_(s, xpositions=x)


def test_large_grid_of_parts(clm):
    """320000 parts of dense cells: the pairs per distance are those of the union-row sweep, which
    takes whole cells."""
    import torch
    side, n = 400.0, 14_000_000
    print(f"[grids] parts n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand((n, 2), generator=g, device="cuda") * side
    s = clm.ParticleSystem(xpositions=x, unitcell=[side] * 2, cutoff=1.0)
    h = clm.pairwise_(clm.DistanceHistogram(16, 1.0 / 16), s)
    s.set_sweep_variant(0)
    assert np.array_equal(h, clm.pairwise_(clm.DistanceHistogram(16, 1.0 / 16), s))
    assert abs(h.sum() / (0.5 * n * n * np.pi / side ** 2) - 1) < 1e-3
