"""Two sets: the forces of every particle of either set, energies, and sums of radial velocities,
with whole cells and with cells in parts, against float64 sums over the oracle's pairs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

UNIT = {np.float32: 2.0 ** -24, np.float64: 2.0 ** -53}


def cells(side):
    return {"ortho": np.array([1.1, 0.9, 1.0]) * side, "open": None,
            "tric": np.array([[1.0, 0.2, 0.1], [0.0, 0.95, 0.15], [0.0, 0.0, 1.0]]) * side}


def points(side, uc, n, seed):
    f = np.random.default_rng(seed).random((n, 3))
    if uc is None:
        return f * side
    return f * uc if uc.ndim == 1 else f @ uc.T


def nearest(uc, v):
    if uc is None:
        return v
    m = np.diag(uc) if uc.ndim == 1 else uc
    f = v @ np.linalg.inv(m).T
    return (f - np.round(f)) @ m.T


# (n, ny, side in cutoffs): cells in parts (the two densest), whole ones, small systems
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric", "open"])
@pytest.mark.parametrize("n,ny,side", [(20_000, 700, 4.6), (20_001, 3_000, 3.9), (20_100, 2_000, 11.0), (700, 20_000, 4.6),
                                       (900, 1_100, 5.0)])
def test_two_set_forces_and_velocities(clm, O, n, ny, side, kind, dtype):
    print(f"[two sets] values n={n} ny={ny} side={side} {kind} {np.dtype(dtype).name}", flush=True)
    u = UNIT[dtype]
    uc = cells(side)[kind]
    if uc is not None:
        uc = uc.astype(dtype).astype(np.float64)
    x, y = points(side, uc, n, n).astype(dtype), points(side, uc, ny, ny + 1).astype(dtype)
    rng = np.random.default_rng(ny)
    vx, vy = rng.normal(size=(n, 3)).astype(dtype), rng.normal(size=(ny, 3)).astype(dtype)
    x64, y64 = x.astype(np.float64), y.astype(np.float64)

    def pairs(cutoff, t, a, b):
        if uc is None:
            return O.pairs_cross(O.make_nonperiodic_box(np.concatenate([a, b]), cutoff, dtype=t), a, b, 1)
        return O.pairs_cross(O.make_box(uc, cutoff, dtype=t), a, b, 1)

    i, j, _, d = pairs(1.0, dtype, x, y)
    r = nearest(uc, x64[i] - y64[j])
    # coordinates below 8 carry errors of a few units of 8: pairs that near to the cutoff may be
    # taken from one side only, and the forces of their particles are left out
    margin = 200 * u
    wide = pairs(1.0 + margin, np.float64, x64, y64)
    edge = wide[3] >= 1.0 - margin
    keep = np.ones(n + ny, bool)
    keep[wide[0][edge]] = keep[n + wide[1][edge]] = False

    eps, sigma = 0.2, 0.7
    inv = 1.0 / ((r * r).sum(1) + 1.0)
    s3 = (sigma * sigma * inv) ** 3
    energy = float((eps * (s3 * s3 - s3)).sum())
    g = (2 * eps * (6 * s3 * s3 - 3 * s3) * inv)[:, None] * r
    f = np.zeros((n + ny, 3))
    np.add.at(f, i, g)
    np.add.at(f, n + j, -g)
    size = np.zeros(n + ny)
    np.add.at(size, i, np.abs(g).sum(1) + eps)
    np.add.at(size, n + j, np.abs(g).sum(1) + eps)
    count = np.bincount(i, minlength=n).max() + np.bincount(j, minlength=ny).max()

    s = clm.ParticleSystem(xpositions=x, ypositions=y, unitcell=uc, cutoff=1.0)
    width = 0.125
    bins = np.minimum(np.floor(d.astype(dtype) / dtype(width)), 7).astype(int)
    dv = vx.astype(np.float64)[i] - vy.astype(np.float64)[j]
    want, bound = np.zeros(8), np.zeros(8)
    np.add.at(want, bins, (dv * r).sum(1) / d)
    # the pair's vector is off by up to 100 units, the term and its distance by a few of their own
    np.add.at(bound, bins, np.abs(dv).sum(1) * (100 * u / np.maximum(d, 1e-3) + 16 * u))
    for turn in range(2):
        h = clm.pairwise_(clm.PairwiseVelocities(8, width, vx, vy), s)
        assert np.array_equal(h.counts, np.bincount(bins, minlength=8))
        assert (np.abs(h.vsum - want) <= bound).all()
        q = clm.pairwise_(clm.SoftCoreEnergyForces(eps, sigma), s)
        e = clm.pairwise_(clm.SoftCoreEnergy(eps, sigma), s)
        # each term within 200 units, and as much again for every addition of a particle's sum
        tol = (200 + count) * u
        assert np.abs(q.forces - f)[keep].max(initial=0) <= tol * size.max()
        assert abs(q.energy - energy) <= tol * eps * len(i) and abs(e.energy - energy) <= tol * eps * len(i)
        clm.update_(s, xpositions=x, ypositions=y)
