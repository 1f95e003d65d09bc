"""The library's host code on a HIP runtime without a GPU (fake_hip.cpp): which kernels a call
launches, with which arguments, on which device and memory, and what it answers.  Every scenario
runs in a process of its own, with the fake runtime loaded before the library."""
import ctypes as C
import importlib.util
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "celllistmap.jl_amd")
HIP = os.environ.get("ROCM_PATH", "/opt/rocm")
SCENARIOS = {}


def scenario(f):
    SCENARIOS[f.__name__] = f
    return f


class Runtime:
    """The fake runtime, the library on top of it, and calls of its C ABI."""

    def __init__(self, fake):
        self.fake = C.CDLL(fake, mode=C.RTLD_GLOBAL)
        self.fake.fake_allocated.restype = C.c_size_t
        self.fake.fake_launch.restype = C.c_char_p
        self.fake.fake_word.restype = C.c_void_p
        spec = importlib.util.spec_from_file_location("clm_lib", os.path.join(PKG, "_lib.py"))
        self.abi = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(self.abi)
        self.L = self.abi.lib()

    def context(self, n=500, device=0, side=8.0, seed=0):
        p = C.c_void_p()
        assert self.L.clm_create(C.byref(p), device, self.abi.CLM_F32, 3) == 0
        self.box(p, side)
        if n:
            self.positions(p, n)
        return p

    def box(self, c, side):
        cell = (np.eye(3) * side).copy()
        assert self.L.clm_set_box(c, ptr(cell), self.abi.ORTHORHOMBIC, 1.0, 1) == 0

    def positions(self, c, n, y=False):
        x = np.random.default_rng(n).random((n, 3)).astype(np.float32)
        return (self.L.clm_set_positions_y if y else self.L.clm_set_positions)(c, ptr(x), n, 0)

    def forces(self, c, n=500):
        p = self.potential()
        e = C.c_double()
        f = np.empty((n, 3), np.float32)
        return self.L.clm_energy_forces(c, C.byref(p), C.byref(e), ptr(f), 0, None)

    def potential(self):
        p = self.abi.SoftCore()
        p.eps[0], p.sigma[0] = 0.2, 0.5
        return p

    def capture(self, c):
        p = self.potential()
        return self.L.clm_graph_capture_energy_forces(c, C.byref(p), None)

    def words(self, part):
        """The watched words of the last launch of a kernel."""
        k = max(k for k in range(self.fake.fake_launches()) if part in self.fake.fake_launch(k).decode())
        out = []
        while len(out) < 64:
            out.append(self.fake.fake_word(k, len(out)))
        return out

    def launched(self):
        """The kernels launched since the last call."""
        names = [self.fake.fake_launch(k).decode() for k in range(self.fake.fake_launches())]
        self.fake.fake_clear_log()
        return names


def ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def first(names, part):
    return next((k for k, v in enumerate(names) if part in v), None)


@scenario
def capture_then_eager(rt):
    """Capturing gives a short list more room: what it held is gone, and a call made before the
    first replay builds it again before it is walked."""
    for op in ("forces", "list"):
        c = rt.context()
        assert rt.forces(c) == 0
        assert rt.capture(c) == 0
        rt.launched()
        if op == "forces":
            assert rt.forces(c) == 0
        else:
            n, buf = C.c_int64(), np.zeros(3000, np.float32)
            assert rt.L.clm_neighborlist(c, ptr(buf), ptr(buf), ptr(buf), 1000, C.byref(n), 1) == 0
        names = rt.launched()
        assert first(names, "k_cell_sort") is not None, names
        assert first(names, "k_cell_sort") < first(names, "k_sweep"), names
        # the list now has its room: the next capture leaves it as it is
        assert rt.capture(c) == 0
        rt.launched()
        assert rt.forces(c) == 0
        assert first(rt.launched(), "k_cell_sort") is None


@scenario
def two_pass_graph_checks_its_build(rt):
    """A graph that bins in two passes (buckets for 9 million cells would take more than 1 GiB)
    hands the build's status block to its sweep, as one that bins in one pass does."""
    rt.fake.fake_watch(b"k_bin_count", 8, 1)
    rt.fake.fake_watch(b"k_sweep_win", 4, 18)
    c = rt.context(side=206.0)
    assert rt.forces(c) == 0
    rt.launched()
    assert rt.capture(c) == 0
    status = rt.words("k_bin_count")[0]
    assert status and status in rt.words("k_sweep_win")
    # an eager two-pass build has read its status before the sweep
    rt.launched()
    assert rt.positions(c, 500) == 0 and rt.forces(c) == 0
    assert status not in rt.words("k_sweep_win")


@scenario
def failed_calls_leave_no_build_to_judge(rt):
    """x's build of a two-set system is left to be checked at the next synchronisation; when y's
    build fails first, the call's error is all that remains: new positions are taken, and the next
    call builds both lists."""
    NAN, OVERFLOW, E_NAN = 1, 4, rt.abi.CLM_ERR_NAN
    for flag in (NAN, OVERFLOW):
        c = rt.context()
        rt.positions(c, 700, y=True)
        assert rt.forces(c, 1200) == 0
        for again in range(2):
            assert rt.positions(c, 500) == 0
            assert rt.positions(c, 701 + again, y=True) == 0  # (another count: y's build reads its status)
            rt.fake.fake_plant(b"k_bin_images", 10, flag)
            rt.fake.fake_plant(b"k_bin_count", 8, NAN)
            assert rt.forces(c, 1300) == E_NAN
            assert rt.positions(c, 500) == 0
            assert rt.positions(c, 701 + again, y=True) == 0
            types = np.zeros(800, np.int32)
            assert rt.L.clm_set_types(c, ptr(types), 500, 0) == 0
            rt.launched()
            assert rt.forces(c, 1300) == 0
            names = rt.launched()
            assert sum("k_cell_sort" in v for v in names) == 2, names
    # either set past its buckets, or with a NaN, where both builds are left to be checked
    for k, flag in ((0, NAN), (1, NAN), (0, OVERFLOW), (1, OVERFLOW)):
        c = rt.context()
        rt.positions(c, 700, y=True)
        assert rt.forces(c, 1200) == 0
        assert rt.positions(c, 500) == 0 and rt.positions(c, 700, y=True) == 0
        if k == 1:
            rt.fake.fake_plant(b"k_bin_images", 10, 0)
        rt.fake.fake_plant(b"k_bin_images", 10, flag)
        assert rt.forces(c, 1200) == (E_NAN if flag == NAN else 0)
        assert rt.positions(c, 500) == 0 and rt.positions(c, 700, y=True) == 0
        assert rt.forces(c, 1200) == 0


@scenario
def refused_calls_leave_no_build_to_judge(rt):
    """A histogram of a batch is refused before anything is built for it."""
    c = rt.context(0)
    n = np.array([200, 300], np.int64)
    cells = np.concatenate([np.eye(3).ravel() * 8.0] * 2)
    cutoffs, lcells = np.ones(2), np.ones(2, np.int32)
    assert rt.L.clm_set_systems(c, 2, ptr(n), ptr(cells), rt.abi.ORTHORHOMBIC, ptr(cutoffs), ptr(lcells)) == 0
    p, e, f = rt.potential(), np.zeros(2), np.empty((500, 3), np.float32)
    for _ in range(2):
        assert rt.positions(c, 500) == 0
        assert rt.L.clm_energy_forces_batch(c, C.byref(p), ptr(e), ptr(f), 0) == 0
    counts = np.zeros(4, np.int64)
    assert rt.positions(c, 500) == 0
    rt.launched()
    assert rt.L.clm_histogram(c, 4, 0.25, ptr(counts), None) == rt.abi.CLM_ERR_ARG
    assert rt.launched() == []
    assert rt.positions(c, 500) == 0


@scenario
def every_call_works_on_its_own_device(rt):
    """Contexts of two devices in one thread: whichever is current, a call allocates, copies and
    launches on its context's device, and what a destroyed context leaves goes to contexts of its
    own device only."""
    rt.fake.fake_devices(2)
    L = rt.L
    types, vel = np.zeros(5000, np.int32), np.zeros((5000, 3), np.float32)
    counts, vsum = np.zeros(4, np.int64), np.zeros(4)
    n, cutoffs, lcells = np.array([2000, 3000], np.int64), np.ones(2), np.ones(2, np.int32)
    cells = np.concatenate([np.eye(3).ravel() * 8.0] * 2)
    info = rt.abi.BoxInfo()
    for turn in range(3):
        made = []
        for device in (0, 1):
            c = rt.context(5000, device)
            rt.positions(c, 5000, y=True)
            o = rt.context(0, device)  # a context that only ever gets a batch
            p = rt.context(5000, device)
            assert L.clm_set_box(p, None, rt.abi.NONPERIODIC, 1.0, 1) == 0
            made.append((c, o, p))
        for device in (0, 1):
            c, o, p = made[device]
            away = lambda: rt.fake.hipSetDevice(1 - device)
            calls = [lambda: L.clm_set_types(c, ptr(types), 5000, 0), lambda: L.clm_set_types_y(c, ptr(types), 5000, 0),
                     lambda: L.clm_set_velocities(c, ptr(vel), 5000, 0), lambda: L.clm_set_velocities_y(c, ptr(vel), 5000, 0),
                     lambda: L.clm_histogram(c, 4, 0.25, ptr(counts), ptr(vsum)), lambda: rt.forces(c, 10000),
                     lambda: L.clm_set_systems(o, 2, ptr(n), ptr(cells), rt.abi.ORTHORHOMBIC, ptr(cutoffs), ptr(lcells)),
                     lambda: rt.positions(o, 5000), lambda: L.clm_get_box(p, C.byref(info)), lambda: rt.forces(p, 5000),
                     lambda: L.clm_clear_positions_y(c), lambda: rt.capture(c)]
            for k, call in enumerate(calls):
                away()
                assert call() == 0, k
                assert rt.fake.fake_misplaced() == 0, k
            for q in made[device]:
                away()
                assert L.clm_destroy(q) == 0


@scenario
def spill_of_a_list_is_bounded(rt):
    """What a list needs beside its own arrays does not grow with the capacity: the spill of 512
    slots to a chunk (33856 chunks of 12 bytes a slot with 5120 waves) with the 25 % that buffers get,
    and three words for every 512 slots of list and spill."""
    spill = 33856 * 512 * 12
    n, out = C.c_int64(), np.zeros(16, np.float32)  # (no kernel runs: nothing is written)
    for cap in (1_000, 1_000_000, 20_000_000, 50_000_000, 200_000_000, 1_000_000_000):
        c = rt.context(200_000, side=40.0)
        assert rt.L.clm_update_cell_list(c) == 0
        before = rt.fake.fake_allocated()
        assert rt.L.clm_neighborlist(c, ptr(out), ptr(out), ptr(out), cap, C.byref(n), 1) == 0
        extra = rt.fake.fake_allocated() - before
        assert extra <= 1.25 * (spill + 12 * (cap + spill // 12) // 512) + (4 << 20), (cap, extra)
        rt.L.clm_destroy(c)


@scenario
def replay_after_a_failed_build(rt):
    """A build with a NaN or an overflow leaves the visiting order without some particles and with
    others twice: a graph that bins in that order is given the particles' own before it runs again;
    eager builds do not use it."""
    rt.fake.fake_watch(b"k_bin_images", 10, 1)
    rt.fake.fake_watch(b"k_bin_count", 8, 1)
    NAN, OVERFLOW = 1, 4
    codes = {NAN: rt.abi.CLM_ERR_NAN, OVERFLOW: rt.abi.CLM_ERR_CAPACITY}
    e = C.c_double()
    for how in ("replay", "eager"):
        for flag in (NAN, OVERFLOW):
            c = rt.context()
            for _ in range(3):
                assert rt.positions(c, 500) == 0 and rt.forces(c) == 0
            assert rt.capture(c) == 0
            status = C.c_uint32.from_address(rt.words("k_bin_images")[0])
            rt.launched()
            assert rt.L.clm_graph_launch(c, C.byref(e)) == 0
            names = rt.launched()
            assert names[0] == "graph", names
            assert rt.positions(c, 500) == 0
            if how == "replay":
                status.value = flag
                assert rt.L.clm_graph_launch(c, C.byref(e)) == codes[flag]
                status.value = 0
            else:
                rt.fake.fake_plant(b"k_bin_images", 10, NAN)
                assert rt.forces(c) == rt.abi.CLM_ERR_NAN
                status.value = 0
            assert rt.positions(c, 500) == 0
            rt.launched()
            assert rt.L.clm_graph_launch(c, C.byref(e)) == 0
            names = rt.launched()
            assert first(names, "k_iota") is not None and first(names, "k_iota") < first(names, "graph"), names
            assert rt.L.clm_graph_launch(c, C.byref(e)) == 0
            assert first(rt.launched(), "k_iota") is None
    # the union-row sweep: the graph bins in two passes and keeps no order, eager builds do
    rt.fake.fake_watch(b"k_bin_images", 2, 1)
    for flag in (NAN, OVERFLOW):
        c = rt.context()
        assert rt.L.clm_set_sweep_variant(c, 0) == 0
        for k in range(3):
            if k:
                rt.fake.fake_plant(b"ProdCells", 6, 500)  # (entries: the sort has something to order)
            assert rt.positions(c, 500) == 0 and rt.forces(c) == 0
        assert rt.words("k_bin_images")[0] is not None
        assert rt.capture(c) == 0
        status = C.c_uint32.from_address(rt.words("k_bin_count")[0])
        status.value = flag
        rt.launched()
        assert rt.L.clm_graph_launch(c, C.byref(e)) == codes[flag]
        status.value = 0
        assert rt.positions(c, 500) == 0 and rt.forces(c) == 0
        assert rt.words("k_bin_images")[0] is None


@scenario
def a_refused_batch_changes_nothing(rt):
    """A batch is refused where there is a second set, and the two-set system goes on as before."""
    c = rt.context()
    rt.positions(c, 700, y=True)
    assert rt.forces(c, 1200) == 0
    n, cutoffs, lcells = np.array([200, 300], np.int64), np.ones(2), np.ones(2, np.int32)
    cells = np.concatenate([np.eye(3).ravel() * 8.0] * 2)
    assert rt.L.clm_set_systems(c, 2, ptr(n), ptr(cells), rt.abi.ORTHORHOMBIC, ptr(cutoffs), ptr(lcells)) == rt.abi.CLM_ERR_ARG
    assert rt.forces(c, 1200) == 0
    assert rt.L.clm_clear_positions_y(c) == 0
    assert rt.positions(c, 400) == 0 and rt.forces(c) == 0


@scenario
def velocities_do_not_outlive_their_particles(rt):
    """More particles than there are velocities: a histogram of radial velocities is refused until
    they are set again (fewer particles take the first of them, as before)."""
    vel, counts, vsum = np.zeros((900, 3), np.float32), np.zeros(4, np.int64), np.zeros(4)
    for y in (False, True):
        c = rt.context()
        if y:
            rt.positions(c, 500, y=True)
            assert rt.L.clm_set_velocities_y(c, ptr(vel), 500, 0) == 0
        assert rt.L.clm_set_velocities(c, ptr(vel), 500, 0) == 0
        hist = lambda: rt.L.clm_histogram(c, 4, 0.25, ptr(counts), ptr(vsum))
        assert hist() == 0
        assert rt.positions(c, 300, y=y) == 0 and hist() == 0
        assert rt.positions(c, 900, y=y) == 0 and hist() == rt.abi.CLM_ERR_STATE
        assert (rt.L.clm_set_velocities_y if y else rt.L.clm_set_velocities)(c, ptr(vel), 900, 0) == 0
        assert hist() == 0


@scenario
def velocities_follow_the_list_they_are_read_with(rt):
    """The velocities of a two-set histogram are laid out along y's entries: whether these may be read
    is said by the status of y's build."""
    rt.fake.fake_watch(b"k_bin_images", 10, 1)
    rt.fake.fake_watch(b"k_entry_velocities", 9, 1)
    vel, counts, vsum = np.zeros((700, 3), np.float32), np.zeros(4, np.int64), np.zeros(4)
    c = rt.context()
    rt.positions(c, 700, y=True)
    assert rt.L.clm_set_velocities(c, ptr(vel), 500, 0) == 0
    assert rt.L.clm_set_velocities_y(c, ptr(vel), 700, 0) == 0
    for turn in range(3):
        rt.positions(c, 500), rt.positions(c, 700, y=True)
        rt.launched()
        assert rt.L.clm_histogram(c, 4, 0.25, ptr(counts), ptr(vsum)) == 0
        if turn:  # (x's status, then y's)
            assert rt.words("k_entry_velocities")[0] == rt.words("k_bin_images")[0]
        else:
            assert rt.words("k_entry_velocities")[0] is None


@scenario
def tuned_group_widths_are_different_kernels(rt):
    """No two of the group widths that the autotuner times by default run the same sweep."""
    spec = importlib.util.spec_from_file_location("autotune", os.path.join(PKG, "autotune.py"))
    autotune = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(autotune)
    c = rt.context(30_000, side=20.0)
    assert rt.forces(c, 30_000) == 0
    sweeps = []
    for group in autotune.GROUPS:
        assert rt.L.clm_set_sweep_group(c, group) == 0
        rt.launched()
        assert rt.capture(c) == 0
        sweeps += [v for v in rt.launched() if "k_sweep" in v]
    assert len(set(sweeps)) == len(autotune.GROUPS) > 1, sweeps


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(os.path.join(HIP, "include", "hip")):
        pytest.skip("no C++ compiler or HIP headers")
    out = tmp_path_factory.mktemp("fake") / "fake_hip.so"
    subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(HIP, "include"),
                    os.path.join(HERE, "fake_hip.cpp"), "-o", str(out)], check=True)
    return str(out)


@pytest.mark.parametrize("name", sorted(SCENARIOS))
def test_host_path(fake, name):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), name, fake], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    SCENARIOS[sys.argv[1]](Runtime(sys.argv[2]))
