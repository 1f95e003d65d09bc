"""Captured graphs and the cell list around them: what an eager call sees between a capture and the
first replay, and what a replay leaves for the calls after it."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CELLS = {"ortho": np.array([8.0, 9.0, 8.5]),
         "tric": np.array([[8.0, 1.6, 0.8], [0.0, 9.0, 1.2], [0.0, 0.0, 8.5]])}
TOL = {np.float32: 1e-4, np.float64: 1e-10}


def say(*a):
    print(*a, flush=True)


def points(uc, n, seed):
    f = np.random.default_rng(seed).random((n, 3))
    return f * uc if uc.ndim == 1 else f @ uc.T


def capture(clm, s):
    p = clm.SoftCoreEnergyForces(0.2, 0.7).params()
    s._ctx.check(s._ctx.lib.clm_graph_capture_energy_forces(s._ctx.ptr, C.byref(p), None), "capture")


def forces(clm, s):
    r = clm.pairwise_(clm.SoftCoreEnergyForces(0.2, 0.7), s)
    return r.energy, r.forces


def close(a, b, dtype):
    return abs(a[0] - b[0]) <= TOL[dtype] * abs(b[0]) and np.linalg.norm(a[1] - b[1]) <= TOL[dtype] * np.linalg.norm(b[1])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric"])
@pytest.mark.parametrize("n", [40, 500])
def test_eager_calls_between_capture_and_replay(clm, n, kind, dtype):
    """A capture gives a short list more room; forces, gradients and lists taken before the first
    replay are those of before the capture."""
    say(f"[graph] eager after capture n={n} {kind} {np.dtype(dtype).name}")
    uc = CELLS[kind]
    s = clm.ParticleSystem(xpositions=points(uc, n, n).astype(dtype), unitcell=uc, cutoff=2.0)
    want = forces(clm, s)
    pairs = clm.neighborlist(xpositions=points(uc, n, n).astype(dtype), unitcell=uc, cutoff=2.0).canonical()
    for op in ("forces", "adjoint", "list"):
        s = clm.ParticleSystem(xpositions=points(uc, n, n).astype(dtype), unitcell=uc, cutoff=2.0)
        forces(clm, s)
        capture(clm, s)
        if op == "forces":
            assert close(forces(clm, s), want, dtype)
        elif op == "adjoint":
            g = clm.energy_adjoint(s, 0.2, 0.7)
            assert close((g.energy, -g.dedx), want, dtype)
        else:
            got = clm.pairwise_(clm.NeighborListOp(), s).canonical()
            assert all(np.array_equal(a, b) for a, b in zip(got, pairs))
        e = C.c_double()
        s._ctx.check(s._ctx.lib.clm_graph_launch(s._ctx.ptr, C.byref(e)), "replay")
        assert abs(e.value - want[0]) <= TOL[dtype] * abs(want[0])
        assert close(forces(clm, s), want, dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric"])
@pytest.mark.parametrize("nsys", [1, 3])
def test_replay_with_nan_in_two_passes(clm, nsys, kind, dtype):
    """A crowded cell in a box of a million: buckets for it would take more than 1 GiB, and the
    graph bins in two passes.  A NaN in any system is reported, and good positions after it give
    what an eager call gives."""
    say(f"[graph] two passes, NaN, nsys={nsys} {kind} {np.dtype(dtype).name}")
    uc = CELLS[kind] / 8.0 * 100.0
    small = CELLS[kind]
    ucs = [uc] + [small] * (nsys - 1)
    xs = []
    for k, u in enumerate(ucs):
        x = points(u, 400, k)
        x[:100] = 0.5 * points(np.ones(3), 100, k + 7) + 40.1 * (k == 0)
        xs.append(x.astype(dtype))
    b = clm.BatchedSystems(xs, ucs, 1.0, lcell=1)
    every = np.concatenate(xs)
    want = b.energy_forces(0.2, 0.7)
    b.capture(0.2, 0.7)
    assert (np.abs(b.replay() - want[0]) <= TOL[dtype] * np.abs(want[0])).all()
    for at in (0, 399, len(every) - 1):
        bad = every.copy()
        bad[at, at % 3] = np.nan
        b.set_positions(bad)
        with pytest.raises(clm.ArgumentError):
            b.replay()
        b.set_positions(every)
        assert (np.abs(b.replay() - want[0]) <= TOL[dtype] * np.abs(want[0])).all()
        b.set_positions(bad)
        with pytest.raises(clm.ArgumentError):
            b.replay()
        b.set_positions(every)
        e, f = b.energy_forces(0.2, 0.7)
        assert (np.abs(e - want[0]) <= TOL[dtype] * np.abs(want[0])).all()
        assert np.linalg.norm(f - want[1]) <= TOL[dtype] * np.linalg.norm(want[1])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["ortho", "tric"])
@pytest.mark.parametrize("variant", [1, 0])
@pytest.mark.parametrize("n", [900, 21_000])
def test_replays_after_a_failed_build(clm, n, variant, kind, dtype):
    """A NaN or a crowded cell in a replay, or a NaN in an eager build between two, is reported; the
    next replay and the next eager call on good positions see every particle once."""
    say(f"[graph] after a failed build n={n} variant={variant} {kind} {np.dtype(dtype).name}")
    uc = CELLS[kind] * (1.0 if n < 20_000 else 2.5)
    x = points(uc, n, n).astype(dtype)
    s = clm.ParticleSystem(xpositions=x, unitcell=uc, cutoff=1.0)
    s.set_sweep_variant(variant)
    for _ in range(2):
        want = forces(clm, s)
        clm.update_(s, xpositions=x)
    capture(clm, s)

    def replay():
        e = C.c_double()
        return s._ctx.lib.clm_graph_launch(s._ctx.ptr, C.byref(e)), e.value

    nan, crowd = x.copy(), x.copy()
    nan[n // 3, 1] = np.nan
    crowd[: n // 2] = 0.3 * crowd[: n // 2] / crowd.max() + 2.0
    E = clm._lib
    for bad, code in ((nan, E.CLM_ERR_NAN), (crowd, E.CLM_ERR_CAPACITY), (None, 0)):
        if bad is None:
            clm.update_(s, xpositions=nan)
            with pytest.raises(clm.ArgumentError):
                forces(clm, s)
        else:
            clm.update_(s, xpositions=bad)
            rc = replay()[0]
            assert rc == code or (code == E.CLM_ERR_CAPACITY and variant == 0 and rc == 0)  # (two passes have no buckets)
        clm.update_(s, xpositions=x)
        for _ in range(2):
            rc, e = replay()
            if rc == E.CLM_ERR_STATE:  # larger buckets since
                capture(clm, s)
                rc, e = replay()
            assert rc == 0 and abs(e - want[0]) <= TOL[dtype] * abs(want[0])
        for bad2 in (nan, x):
            clm.update_(s, xpositions=bad2)
            if bad2 is nan:
                assert replay()[0] == E.CLM_ERR_NAN
            else:
                assert close(forces(clm, s), want, dtype)
