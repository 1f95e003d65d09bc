"""The windowed sweep's task shapes: how many lanes share a particle, and so how many
particles make a task, depends on the number of particles and on the entries of a stencil
row's window.  Systems on both sides of each line, with counts that leave the last task of a
row partly empty, against the oracle: pair sets and distances bit for bit, minimum distances
exact, energies and forces to 1e-10 (float64) or 1e-4 (float32) of the same sums in float64
over the oracle's pairs (which pairs lie within the cutoff is decided in the system's own
precision, and the potential does not vanish there; the two sides of a pair across a box
face decide it from images of their own, so the forces of particles with a pair within
rounding of the cutoff are left out of the comparison)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def cells(dim, side):
    if dim == 2:
        return {"ortho": np.array([1.1, 0.9]) * side,
                "tric": np.array([[1.0, 0.15], [0.0, 0.95]]) * side}
    return {"ortho": np.array([1.1, 0.9, 1.0]) * side,
            "tric": np.array([[1.0, 0.2, 0.1], [0.0, 0.95, 0.15], [0.0, 0.0, 1.0]]) * side}


def points(uc, n, seed):
    f = np.random.default_rng(seed).random((n, uc.shape[0]))
    return f * uc if uc.ndim == 1 else f @ uc.T


def softcore(uc, x, i, j, eps, sigma):
    """Energy and forces of the pairs (i, j) in float64, by the nearest image."""
    m = np.diag(uc) if uc.ndim == 1 else uc
    x = x.astype(np.float64)
    f = (x[i] - x[j]) @ np.linalg.inv(m).T
    v = (f - np.round(f)) @ m.T
    inv = 1.0 / ((v * v).sum(1) + 1.0)
    s3 = (sigma * sigma * inv) ** 3
    g = (2 * eps * (6 * s3 * s3 - 3 * s3) * inv)[:, None] * v
    forces = np.zeros_like(x)
    np.add.at(forces, i, g)
    np.add.at(forces, j, -g)
    return float((eps * (s3 * s3 - s3)).sum()), forces


# (n, dim, side in cutoffs, lcell): the smallest systems, 20000 particles and one either side,
# short windows (below 160 entries) and long ones
SIZES = [(1, 3, 3.2, 1), (2, 3, 3.2, 2), (65, 3, 3.2, 1), (1000, 3, 4.1, 1), (999, 2, 12.3, 2),
         (19_999, 3, 9.3, 2), (20_000, 3, 9.3, 1), (20_001, 3, 5.2, 1), (20_001, 3, 14.0, 3), (33_333, 2, 25.0, 1)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric"])
@pytest.mark.parametrize("n,dim,side,lcell", SIZES)
def test_task_shapes(clm, O, n, dim, side, lcell, kind, dtype):
    rc = 1.0
    uc = cells(dim, side)[kind].astype(dtype).astype(np.float64)
    x = points(uc, n, n + dim + lcell).astype(dtype)
    say(f"[shapes] n={n} dim={dim} side={side} lcell={lcell} {kind} {np.dtype(dtype).name}")
    box = O.make_box(uc, rc, lcell=lcell, dtype=dtype)
    s = clm.ParticleSystem(xpositions=x, unitcell=uc, cutoff=rc, lcell=lcell)
    a, b, d = clm.pairwise_(clm.NeighborListOp(), s).canonical()
    i, j, _, do = O.pairs(box, x, 1)
    lo, hi = np.minimum(i, j), np.maximum(i, j)
    o = np.lexsort((do, hi, lo))
    k = np.lexsort((d, b, a))
    assert np.array_equal(a[k], lo[o]) and np.array_equal(b[k], hi[o])
    assert np.array_equal(d[k].astype(np.float64), do[o])
    if len(do):
        m = clm.pairwise_(clm.MinimumDistance(), s)
        t = np.lexsort((hi, lo, do))[0]
        assert (m[0], m[1]) == (lo[t], hi[t]) and m[2] == do[t]
    h = clm.pairwise_(clm.DistanceHistogram(7, rc / 6), s)
    width, dd = dtype(rc / 6), do.astype(dtype)
    assert np.array_equal(h, np.bincount(np.minimum(np.floor(dd / width), 6).astype(int), minlength=7))
    tol = 1e-10 if dtype == np.float64 else 1e-4
    energy, forces = softcore(uc, x, i, j, 0.2, 0.7)
    near = tol * max(np.linalg.norm(forces), 1e-12)
    # coordinates below 32 carry errors below 4e-6 in float32
    margin = 1e-5 if dtype == np.float32 else 1e-13
    x64 = x.astype(np.float64)
    wide = O.pairs(O.make_box(uc, rc + margin, lcell=lcell), x64, 1)
    edge = wide[3] >= rc - margin
    keep = np.ones(n, bool)
    keep[wide[0][edge]] = keep[wide[1][edge]] = False
    r = clm.pairwise_(clm.SoftCoreEnergyForces(0.2, 0.7), s)
    e = clm.pairwise_(clm.SoftCoreEnergy(0.2, 0.7), s)
    scale = max(abs(energy), 1e-12)
    assert abs(r.energy - energy) <= tol * scale and abs(e.energy - energy) <= tol * scale
    assert np.linalg.norm((r.forces - forces)[keep]) <= near
    g = clm.energy_adjoint(s, 0.2, 0.7)
    assert abs(g.energy - energy) <= tol * scale
    assert np.linalg.norm((g.dedx + forces)[keep]) <= near
    assert abs(g.deps[0] - energy / 0.2) <= tol * scale / 0.2


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric"])
@pytest.mark.parametrize("n,ny,side", [(3, 20_100, 8.0), (20_100, 3, 8.0), (20_100, 2_000, 11.0)])
def test_task_shapes_two_sets(clm, O, n, ny, side, kind, dtype):
    uc = cells(3, side)[kind].astype(dtype).astype(np.float64)
    x, y = points(uc, n, n).astype(dtype), points(uc, ny, ny + 1).astype(dtype)
    say(f"[shapes] two sets n={n} ny={ny} {kind} {np.dtype(dtype).name}")
    box = O.make_box(uc, 1.0, lcell=1, dtype=dtype)
    s = clm.ParticleSystem(xpositions=x, ypositions=y, unitcell=uc, cutoff=1.0)
    a, b, d = clm.pairwise_(clm.NeighborListOp(), s).ordered()
    i, j, _, do = O.pairs_cross(box, x, y, 1)
    o, k = np.lexsort((do, j, i)), np.lexsort((d, b, a))
    assert len(a) and np.array_equal(a[k], i[o]) and np.array_equal(b[k], j[o])
    assert np.array_equal(d[k].astype(np.float64), do[o])
    f = clm.pairwise_(clm.SoftCoreEnergyForces(0.2, 0.7), s).forces
    assert np.linalg.norm(f.sum(0)) <= (1e-10 if dtype == np.float64 else 1e-4) * np.abs(f).sum()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,dim,side,lcell", [(700, 3, 3.1, 1), (19_999, 2, 40.0, 1), (40_001, 3, 22.0, 1),
                                              (110_003, 3, 30.0, 2), (150_001, 2, 120.0, 1), (300_007, 3, 45.0, 1)])
def test_rebuilt_list_is_the_same(clm, O, n, dim, side, lcell, dtype):
    """First builds (two passes, status read) and rebuilds (one pass, status deferred) of cell
    lists of all sizes: the sort takes 4, 2 or 1 threads per entry, the binning a thread per
    particle and image or per particle."""
    uc = cells(dim, side)["ortho"].astype(dtype).astype(np.float64)
    x = points(uc, n, n).astype(dtype)
    say(f"[shapes] rebuild n={n} dim={dim} {np.dtype(dtype).name}")
    nl = clm.InPlaceNeighborList(xpositions=x, unitcell=uc, cutoff=1.0, lcell=lcell)
    i, j, _, do = O.pairs(O.make_box(uc, 1.0, lcell=lcell, dtype=dtype), x, 1)
    lo, hi = np.minimum(i, j), np.maximum(i, j)
    o = np.lexsort((do, hi, lo))
    for k in range(3):
        a, b, d = clm.neighborlist_(nl).canonical()
        assert np.array_equal(a, lo[o]) and np.array_equal(b, hi[o]) and np.array_equal(d.astype(np.float64), do[o])
        clm.update_(nl, xpositions=x)


def in_order(i, j, d):
    """A list by (lower index, higher index), sorted on the GPU (lists of 10^7 pairs)."""
    import torch
    i, j, d = (torch.as_tensor(np.ascontiguousarray(v)).cuda() for v in (i, j, d))
    key, at = torch.sort(torch.minimum(i, j).long() << 32 | torch.maximum(i, j).long())
    return key.cpu().numpy(), d[at].cpu().numpy().astype(np.float64)


# (n, dim, side in cutoffs, lcell): rows of a cell hold enough for 2, 3, 2 and 4 parts
PARTS = [(20_001, 3, 5.2, 1), (20_001, 3, 3.9, 1), (20_001, 3, 3.9, 2), (20_001, 2, 9.0, 1)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric", "open"])
@pytest.mark.parametrize("n,dim,side,lcell", PARTS)
def test_cells_in_parts(clm, O, n, dim, side, lcell, kind, dtype):
    """Dense cells are cut into parts along y and z unless the first operator is a list: the
    same pairs, counts and closest pair as the oracle's whole cells, the reference's cell
    counts, and the same after a switch of the sweep variant and back (another grid each time)."""
    if kind == "open" and lcell > 1:
        pytest.skip("one open box per size")
    uc = cells(dim, side)["tric" if kind == "tric" else "ortho"].astype(dtype).astype(np.float64)
    x = points(uc, n, n + dim).astype(dtype)
    say(f"[parts] n={n} dim={dim} lcell={lcell} {kind} {np.dtype(dtype).name}")
    if kind == "open":
        box = O.make_nonperiodic_box(x, 1.0, lcell=lcell, dtype=dtype)
    else:
        box = O.make_box(uc, 1.0, lcell=lcell, dtype=dtype)
    i, j, _, do = O.pairs(box, x, 1)
    key, dist = in_order(i, j, do)
    t = np.flatnonzero(do == do.min())
    closest = min((min(i[k], j[k]), max(i[k], j[k])) for k in t) + (do.min(),)
    s = clm.ParticleSystem(xpositions=x, unitcell=None if kind == "open" else uc, cutoff=1.0, lcell=lcell)
    counts = np.bincount(np.minimum(np.floor(do.astype(dtype) / dtype(0.125)), 7).astype(int), minlength=8)
    stats = O.cl_stats(box, x)
    for variant in (1, 0, 1):
        s.set_sweep_variant(variant)
        assert np.array_equal(clm.pairwise_(clm.DistanceHistogram(8, 0.125), s), counts)
        assert s.cell_list_info() == stats
        assert clm.pairwise_(clm.MinimumDistance(), s) == closest
        r = clm.pairwise_(clm.NeighborListOp(), s)
        k, d = in_order(r.i, r.j, r.d)
        assert np.array_equal(k, key) and np.array_equal(d, dist)
        clm.update_(s, xpositions=x)
    if dtype == np.float64:
        ref = O.softcore(box, x, eps=0.2, sigma=0.5)
        for _ in range(2):
            r = clm.pairwise_(clm.SoftCoreEnergyForces(0.2, 0.5), s)
            assert abs(r.energy - ref["energy"]) <= 1e-10 * abs(ref["energy"])
            assert np.linalg.norm(r.forces - ref["forces"]) <= 1e-10 * np.linalg.norm(ref["forces"])
            clm.update_(s, xpositions=x)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric"])
def test_cells_in_parts_two_sets_and_batch(clm, O, kind, dtype):
    uc = cells(3, 4.6)[kind].astype(dtype).astype(np.float64)
    x, y = points(uc, 20_000, 1).astype(dtype), points(uc, 700, 2).astype(dtype)
    say(f"[parts] two sets and batch {kind} {np.dtype(dtype).name}")
    box = O.make_box(uc, 1.0, dtype=dtype)
    i, j, _, do = O.pairs_cross(box, x, y, 1)
    s = clm.ParticleSystem(xpositions=x, ypositions=y, unitcell=uc, cutoff=1.0)
    counts = np.bincount(np.minimum(np.floor(do.astype(dtype) / dtype(0.125)), 7).astype(int), minlength=8)
    for _ in range(2):
        assert np.array_equal(clm.pairwise_(clm.DistanceHistogram(8, 0.125), s), counts)
        clm.update_(s, ypositions=y)
    a, b, d = clm.pairwise_(clm.NeighborListOp(), s).ordered()
    o = np.lexsort((do, j, i))
    assert np.array_equal(a, i[o]) and np.array_equal(b, j[o]) and np.array_equal(d.astype(np.float64), do[o])
    # a batch of a dense, a sparse and a tiny system: each cut (or not) by its own density
    sizes, sides = [22_000, 900, 40], [4.6, 6.0, 3.0]
    ucs = [cells(3, v)[kind] for v in sides]
    xs = [points(u, m, m) for u, m in zip(ucs, sizes)]
    bt = clm.BatchedSystems([v.astype(dtype) for v in xs], ucs, 1.0, lcell=1)
    e, f = bt.energy_forces(0.2, 0.5)
    bt.capture(0.2, 0.5)
    again = bt.replay()
    tol = 1e-10 if dtype == np.float64 else 1e-4
    for k in range(3):
        ref = O.softcore(O.make_box(ucs[k], 1.0), xs[k], eps=0.2, sigma=0.5)
        assert abs(e[k] - ref["energy"]) <= tol * abs(ref["energy"]) and abs(again[k] - ref["energy"]) <= tol * abs(ref["energy"])
        if dtype == np.float64:
            assert np.linalg.norm(bt.split(f)[k] - ref["forces"]) <= tol * np.linalg.norm(ref["forces"])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric", "open"])
@pytest.mark.parametrize("n,side,lcell", [(900, 4.2, 4), (20_003, 16.0, 5)])
def test_many_rows(clm, O, n, side, lcell, kind, dtype):
    """Stencils of 81 and 121 rows, most of them empty of entries or of windows: the rows of a
    particle take several lists of windows, and lists may be empty."""
    uc = cells(3, side)["ortho" if kind == "open" else kind].astype(dtype).astype(np.float64)
    x = points(uc, n, lcell).astype(dtype)
    say(f"[shapes] rows n={n} lcell={lcell} {kind} {np.dtype(dtype).name}")
    cell = None if kind == "open" else uc
    s = clm.ParticleSystem(xpositions=x, unitcell=cell, cutoff=1.0, lcell=lcell)
    a, b, d = clm.pairwise_(clm.NeighborListOp(), s).canonical()
    if kind == "open":
        box = O.make_nonperiodic_box(x, 1.0, lcell=lcell, dtype=dtype)
    else:
        box = O.make_box(uc, 1.0, lcell=lcell, dtype=dtype)
    i, j, _, do = O.pairs(box, x, 1)
    lo, hi = np.minimum(i, j), np.maximum(i, j)
    o, k = np.lexsort((do, hi, lo)), np.lexsort((d, b, a))
    assert np.array_equal(a[k], lo[o]) and np.array_equal(b[k], hi[o])
    assert np.array_equal(d[k].astype(np.float64), do[o])
    h = clm.pairwise_(clm.DistanceHistogram(7, 1.0 / 6), s)
    assert np.array_equal(h, np.bincount(np.minimum(np.floor(do.astype(dtype) / dtype(1.0 / 6)), 6).astype(int), minlength=7))


@pytest.mark.parametrize("velocity", [0.0, 1e-44, 1e-30, 1.5, 3e37, np.inf])
def test_histogram_bins_and_radial_velocity(clm, velocity):
    """Float32 distances on and next to bin edges, and radial velocities of any size: the counts
    of floor(d / width) with root and quotient rounded, and v.r / d to 4 units of 2^-24 (one for
    the quotient, two for a distance an ulp off) and one of the smallest float."""
    f = np.float32
    width = f(0.1)
    k = np.arange(1, 40)
    edge = (k.astype(f) * width).astype(f)
    steps = [np.nextafter(edge, f(0)), edge, np.nextafter(edge, f(10)), (edge * f(1.37)).astype(f)]
    for dist in steps:
        dist = np.concatenate([dist[dist < f(4)], f([1e-3, 1e-17, 1e-22])])
        # pairs far from each other along y, each of two particles `dist` apart along x
        m = len(dist)
        x = np.zeros((2 * m, 3), f)
        x[0::2, 1] = x[1::2, 1] = 10 * np.arange(m)
        x[1::2, 0] = dist
        v = np.zeros((2 * m, 3), f)
        v[1::2, 0] = f(velocity)
        with np.errstate(all="ignore"):
            d2 = (x[1::2, 0] - x[0::2, 0]) ** 2 + f(0)
            d = np.sqrt(d2)
            t = (v[1::2, 0] - v[0::2, 0]) * (x[1::2, 0] - x[0::2, 0])
            radial = np.where(d > 0, (t / np.where(d > 0, d, f(1))).astype(np.float64), 0.0)
        bins = np.minimum(np.floor(d / width), 39).astype(int)
        s = clm.ParticleSystem(xpositions=x, unitcell=None, cutoff=4.0)
        h = clm.pairwise_(clm.PairwiseVelocities(40, float(width), v), s)
        assert np.array_equal(h.counts, np.bincount(bins, minlength=40))
        want = np.zeros(40)
        size = np.zeros(40)
        with np.errstate(all="ignore"):
            np.add.at(want, bins, radial)
            np.add.at(size, bins, np.abs(radial))
            ok = np.isfinite(want)
            assert np.array_equal(h.vsum[~ok], want[~ok])
            assert (np.abs(h.vsum - want)[ok] <= 4 * 2.0 ** -24 * size[ok] + np.bincount(bins, minlength=40)[ok] * 2.0 ** -149).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,n,ny", [(3, 1, 0), (2, 255, 0), (3, 257, 0), (3, 31_000, 0), (2, 40_001, 0), (3, 300, 70_000)])
def test_limits_of_an_open_box(clm, O, dim, n, ny, dtype):
    """The open box is laid over the exact extremes of the coordinates, wherever they stand
    among the particles and in either set; a NaN anywhere is refused."""
    rng = np.random.default_rng(n + ny + dim)
    x = (rng.random((n, dim)) * 3 - 7).astype(dtype)
    y = (rng.random((ny, dim)) * 3 - 7).astype(dtype) if ny else None
    every = x if y is None else np.concatenate([x, y])
    last = every.shape[0] - 1
    for at, value in ((0, -9.25), (last, 11.5), (last // 2, -9.5)):
        part, k = (x, at) if at < n else (y, at - n)
        part[k, at % dim] = value
    every = x if y is None else np.concatenate([x, y])
    s = clm.ParticleSystem(xpositions=x, ypositions=y, unitcell=None, cutoff=0.5)
    d = np.diag(np.asarray(s.box["input"]).reshape(dim, dim))
    want = (every.max(0) - every.min(0)) + dtype(210) * dtype(0.5) / dtype(100)
    assert np.array_equal(d.astype(dtype), want)
    bad = (x if y is None else y).copy()
    bad[-1, dim - 1] = np.nan
    # (the check of the coordinates on the host is off: the device finds it)
    with pytest.raises(clm.ArgumentError):
        if y is None:
            t = clm.ParticleSystem(xpositions=bad, unitcell=None, cutoff=0.5, validate_coordinates=None)
        else:
            t = clm.ParticleSystem(xpositions=x, ypositions=bad, unitcell=None, cutoff=0.5, validate_coordinates=None)
        clm.pairwise_(clm.MinimumDistance(), t)
