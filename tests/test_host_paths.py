"""The library's host code without a GPU: libvrh with a test double of the HIP
runtime (hip_double.cpp) loaded before it, each case in a process of its own.
Copies, events and streams behave; kernels are counted and compute nothing."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = """
import ctypes, os, threading
import numpy as np
dbl = ctypes.CDLL(os.environ["HIP_DOUBLE"])
import vring_amd
"""


@pytest.fixture(scope="session")
def double(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "hip_double.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    os.path.join(HERE, "hip_double.cpp"), "-o", so, "-lpthread"], check=True)
    return so


@pytest.fixture
def run(double):
    def go(body):
        env = dict(os.environ)
        env["HIP_DOUBLE"] = double
        env["LD_PRELOAD"] = " ".join(filter(None, [double, env.get("LD_PRELOAD", "")]))
        env["PYTHONPATH"] = os.pathsep.join(filter(None, [os.path.dirname(HERE), env.get("PYTHONPATH", "")]))
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body)], env=env, capture_output=True,
                           text=True, timeout=120)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return go


def test_downloads_of_one_handle_in_threads(run):
    """Two threads that fetch different fields of one idle handle each get
    their own: results of 9 MB go through the handle's staging memory."""
    run("""
    nt, nr, nz = 64, 61, 270
    s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01)
    want = {n: np.random.default_rng(q).standard_normal((nt, nr + 3, nz + 3)) for q, n in enumerate(("q1", "q2", "q3"))}
    for n, a in want.items():
        s.upload(n, a)
    bad = []
    def work(n):
        for _ in range(4):
            if not np.array_equal(s.download(n), want[n]):
                bad.append(n)
    th = [threading.Thread(target=work, args=(n,)) for n in want]
    [t.start() for t in th]
    [t.join() for t in th]
    assert not bad, bad
    """)


def test_download_beside_other_work_on_the_field(run):
    """A large result is the field at one point of the handle's stream, also
    while another thread keeps writing the field."""
    run("""
    nt, nr, nz = 64, 61, 270
    s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01)
    vals = [np.full((nt, nr + 3, nz + 3), float(k)) for k in range(4)]
    s.upload("q1", vals[0])
    stop = threading.Event()
    def write():
        k = 0
        while not stop.is_set():
            k += 1
            s.upload("q1", vals[k % 4])
    t = threading.Thread(target=write)
    t.start()
    try:
        mixed = sum(len(np.unique(s.download("q1"))) != 1 for _ in range(10))
    finally:
        stop.set()
        t.join()
    assert mixed == 0, mixed
    """)


def test_particle_download_needs_no_device_memory(run):
    """A batch's particles come down also where the device has no memory left
    (by the host alone), and the next download takes the device's rows."""
    run("""
    s = vring_amd.Solver(8, 8, 8, 4.0, 12.0, 1000.0, 0.01)
    s.particles_create([1000], st=[0.0], nsub=[1], scheme="trilinear_rk3")
    dbl.dbl_fail(ctypes.c_long(-1), ctypes.c_long(0))
    dbl.dbl_reset()
    u, alive = s.particles_download(0, 1000)
    assert u.shape == (1000, 6) and not u.any() and not alive.any()
    assert dbl.dbl_runs(b"k_rows_out") == 0
    dbl.dbl_fail(ctypes.c_long(0), ctypes.c_long(0))
    s.particles_download(0, 1000)
    assert dbl.dbl_runs(b"k_rows_out") == 1
    """)


def test_first_large_downloads_make_no_staging(run):
    """The pinned slots take longer to make than one large download gains: a
    handle makes them once it has fetched 64 MB, a result of 32 MB at once."""
    run("""
    def pinned():
        return dbl.dbl_pinned()
    s = vring_amd.Solver(64, 61, 270, 4.0, 12.0, 1000.0, 0.01)   # 9 MB a field
    p0 = pinned()
    a = np.random.default_rng(0).standard_normal((64, 64, 273))
    s.upload("q1", a)
    for n in range(7):
        assert np.array_equal(s.download("q1"), a) and pinned() == p0, n
    assert np.array_equal(s.download("q1"), a) and pinned() == p0 + (8 << 20)
    s = vring_amd.Solver(64, 125, 653, 4.0, 12.0, 1000.0, 0.01)  # 43 MB a field
    p0 = pinned()
    s.download("q1")
    assert pinned() == p0 + (8 << 20)
    """)


@pytest.mark.parametrize("nt,nr,nz,kernel", [(32, 24, 64, "k_dctz2"), (12, 24, 20, "k_zdense2")])
def test_tuned_mixed_steps_share_the_low_modes_launches(run, nt, nr, nz, kernel):
    """A chosen width of the z transforms (by the tuner or by hand) leaves a
    small mixed grid its shared launches: six z transforms a step, no others."""
    run(f"""
    for tune in (lambda s: None, lambda s: s.autotune(), lambda s: s.set_tuning(dct_lines=8)):
        s = vring_amd.Solver({nt}, {nr}, {nz}, 4.0, 12.0, 1000.0, 0.01, precision="mixed")
        tune(s)
        dbl.dbl_reset()
        s.step(2)
        assert dbl.dbl_runs(b"{kernel}") == 12 and dbl.dbl_runs(b"k_radial2") == 6
        assert dbl.dbl_runs(b"k_dctz") + dbl.dbl_runs(b"k_zdense") == 12 and dbl.dbl_refused() == 0
    """)


@pytest.mark.parametrize("what", ["allocation", "copy"])
def test_failed_axial_mesh_leaves_the_previous_one(run, what):
    """vrh_set_axial_mesh on a handle that steps on another mesh, with each of
    its allocations or copies failing in turn: the call reports it, the next
    steps run on the old mesh's matrices and metric and on no freed memory."""
    run(f"""
    import sys
    sys.path.insert(0, {HERE!r})
    from oracle_lib import tanh_axial_mesh
    nt, nr, nz = 8, 8, 16
    dbl.dbl_given.restype = ctypes.c_void_p
    def given(kernel, n):
        return np.copy(np.ctypeslib.as_array(ctypes.cast(dbl.dbl_given(kernel), ctypes.POINTER(ctypes.c_double)), (n,)))
    def used():
        dbl.dbl_reset()
        s.step(1)
        return given(b"k_project", 7 * (nz + 3)), given(b"k_zdense", 64)
    s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01)
    s.set_axial_mesh(*tanh_axial_mesh(nz, 12.0, 2.0))
    s.step(20)
    old = used()
    n = failed = 0
    while True:
        n += 1
        dbl.dbl_fail(ctypes.c_long(n if {what!r} == "allocation" else 0), ctypes.c_long(n if {what!r} == "copy" else 0))
        try:
            s.set_axial_mesh(*tanh_axial_mesh(nz, 12.0, 3.0))
            done = True
        except RuntimeError:
            done = False
        dbl.dbl_fail(ctypes.c_long(0), ctypes.c_long(0))
        now = used()
        assert dbl.dbl_dead() == 0, n
        if done:
            break
        failed += 1
        assert all(np.array_equal(a, b) for a, b in zip(old, now)), n
    assert failed >= 2 and not np.array_equal(old[0], now[0])
    """)


def test_first_steps_on_an_axial_mesh_are_launched_one_by_one(run):
    """Capturing a step takes longer than the first few steps on a mesh gain."""
    run(f"""
    import sys
    sys.path.insert(0, {HERE!r})
    from oracle_lib import tanh_axial_mesh
    s = vring_amd.Solver(8, 8, 16, 4.0, 12.0, 1000.0, 0.01)
    for stretch in (2.0, 3.0):
        s.set_axial_mesh(*tanh_axial_mesh(16, 12.0, stretch))
        dbl.dbl_reset()
        for _ in range(8):
            s.step(1)
        assert dbl.dbl_graphs() == 0 and dbl.dbl_runs(b"k_project") == 24
        s.step(1)
        s.step(3)
        assert dbl.dbl_graphs() == 1 and dbl.dbl_runs(b"k_project") == 36
    s.set_axial_mesh(*tanh_axial_mesh(16, 12.0, 2.0))
    dbl.dbl_reset()
    s.step(20)
    assert dbl.dbl_graphs() == 1 and dbl.dbl_runs(b"k_project") == 60
    """)


@pytest.mark.parametrize("nz", [300, 320, 321])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("refused", [False, True])
def test_dense_z_transforms_fit_the_lds_granted(run, nz, precision, refused):
    """Tiles of 32 lines of 257 to 320 points take more than 64 KB; without the
    device's consent to that a grid with such lines keeps tiles of 16."""
    big = 32 * 8 * nz if nz <= 320 and not refused else 16 * 8 * nz
    run(f"""
    dbl.dbl_refuse_lds({int(refused)})
    s = vring_amd.Solver(64, 128, {nz}, 4.0, 12.0, 1000.0, 0.01, precision={precision!r})
    dbl.dbl_reset()
    s.step(1)
    assert dbl.dbl_refused() == 0 and dbl.dbl_lds(b"k_zdense") == {big}, (dbl.dbl_refused(), dbl.dbl_lds(b"k_zdense"))
    """)


@pytest.mark.parametrize("nt,nr,nz", [(16, 16, 16), (64, 64, 300)])
def test_pressure_solves_of_one_handle_in_threads(run, nt, nr, nz):
    """Each thread's solve has the handle's array to itself until its result is
    out (no kernel computes here: the result is the right-hand side)."""
    run(f"""
    s = vring_amd.Solver({nt}, {nr}, {nz}, 4.0, 12.0, 1000.0, 0.01)
    bad = []
    def work(q):
        rhs = np.asfortranarray(np.random.default_rng(q).standard_normal(({nt}, {nr}, {nz})))
        for _ in range(8):
            if not np.array_equal(s.poisson(rhs), rhs):
                bad.append(q)
    th = [threading.Thread(target=work, args=(q,)) for q in range(3)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert not bad, bad
    """)


def test_failed_chunk_is_reported_as_itself(run):
    """Any of a staged download's copies failing: the call returns -3 with the
    failure's own error, and the next download is whole."""
    run("""
    dbl.hipGetErrorString.restype = ctypes.c_char_p
    s = vring_amd.Solver(64, 125, 653, 4.0, 12.0, 1000.0, 0.01)
    a = np.random.default_rng(0).standard_normal((64, 128, 656))
    s.upload("q1", a)
    for n in (1, 2, 5, 17, 42):
        dbl.dbl_fail(ctypes.c_long(0), ctypes.c_long(n))
        try:
            s.download("q1")
            raise SystemExit(f"copy {n} not reported")
        except RuntimeError as e:
            assert "(-3)" in str(e) and "error 1" in str(e), e
        assert np.array_equal(s.download("q1"), a), n
    """)
