"""Two-set systems whose later builds, left to be checked at the next synchronisation, hold a NaN or
outgrow their cells' buckets in either set: the call reports it or runs again, and the step after it
is right (against the oracle: pairs and distances bit for bit)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CELLS = {"ortho": np.array([6.0, 6.6, 5.4]),
         "tric": np.array([[6.0, 1.2, 0.6], [0.0, 5.7, 0.9], [0.0, 0.0, 6.0]])}


def say(*a):
    print(*a, flush=True)


def points(uc, n, seed):
    f = np.random.default_rng(seed).random((n, 3))
    return f * uc if uc.ndim == 1 else f @ uc.T


def check(clm, O, s, box, x, y):
    i, j, _, d = O.pairs_cross(box, x, y, 1)
    o = np.lexsort((d, j, i))
    a, b, e = clm.pairwise_(clm.NeighborListOp(), s).ordered()
    k = np.lexsort((e, b, a))
    assert np.array_equal(a[k], i[o]) and np.array_equal(b[k], j[o]) and np.array_equal(e[k].astype(np.float64), d[o])
    m = clm.pairwise_(clm.MinimumDistance(), s)
    t = np.lexsort((j, i, d))[0]
    assert (m[0], m[1], m[2]) == (i[t], j[t], d[t])


OPS = {"closest": lambda clm, s: clm.pairwise_(clm.MinimumDistance(), s),
       "list": lambda clm, s: clm.pairwise_(clm.NeighborListOp(), s),
       "forces": lambda clm, s: clm.pairwise_(clm.SoftCoreEnergyForces(0.2, 0.5), s)}


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric"])
@pytest.mark.parametrize("where", ["x", "y", "xy"])
@pytest.mark.parametrize("op", sorted(OPS))
def test_step_after_a_failed_build(clm, O, op, where, kind, dtype):
    say(f"[two sets] {op} {where} {kind} {np.dtype(dtype).name}")
    uc = CELLS[kind].astype(dtype).astype(np.float64)
    box = O.make_box(uc, 1.0, dtype=dtype)
    x, y = points(uc, 800, 1).astype(dtype), points(uc, 900, 2).astype(dtype)
    s = clm.ParticleSystem(xpositions=x, ypositions=y, unitcell=uc, cutoff=1.0)
    check(clm, O, s, box, x, y)
    for fault in ("nan", "crowd"):
        for ny in (900, 850, 900):  # (another count of y reads the status of y's build before x's)
            y = points(uc, ny, ny + 1).astype(dtype)
            bx, by = x.copy(), y.copy()
            for name, v in (("x", bx), ("y", by)):
                if name in where:
                    if fault == "nan":
                        v[len(v) // 2, 1] = np.nan
                    else:
                        v[:600] = (0.3 * v[:600] / 6.0 + 2.0).astype(dtype)
            clm.update_(s, xpositions=bx, ypositions=by)
            if fault == "nan":
                with pytest.raises(clm.ArgumentError):
                    OPS[op](clm, s)
            else:
                OPS[op](clm, s)
                check(clm, O, s, box, bx, by)
            clm.update_(s, xpositions=x, ypositions=y)
            check(clm, O, s, box, x, y)
