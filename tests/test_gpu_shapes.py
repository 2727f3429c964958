"""The substep at the edges of the rules that pick its kernels from the grid:
theta lengths around the explicit kernels' row widths (32 and 64 lanes, 2, 3
and 4 cells a lane) in every form, and the segment lengths of the grouped r
and z sweeps, with and without lanes and waves to spare, against the single
sweeps' results and the oracle."""
import numpy as np
import pytest

import vring_amd
from gpu_common import compare, make_pair, seed_fields, seed_random

pytestmark = pytest.mark.gpu


def substeps(o, s):
    """To the 1e-11 of the other phase tests."""
    for irk in (1, 2, 3):
        for p in ["ucoeff", "coesys", "hdnbc", "hdnl1", "hdnl2", "hdnl3", "step"]:
            assert o.phase(p, irk) == 0
        for p in ["hdnbc", "explicit", "adi"]:
            s.phase(p, irk)
        compare(o, s, ["dq1", "dq2", "dq3", "ru1", "ru2", "ru3"], 1e-11)
        for p in ["divq", "laplace", "upsol", "uppres"]:
            assert o.phase(p, irk) == 0
        for p in ["poisson", "project"]:
            s.phase(p, irk)
        compare(o, s, ["dph", "q1", "q2", "q3", "pres", "prg"], 1e-11)


@pytest.mark.parametrize("nt", [4, 31, 32, 63, 64, 65, 127, 129, 191, 192, 193, 255, 256])
@pytest.mark.parametrize("form", [-1, 0, 1, 2, 3])
def test_explicit_row_widths_match_oracle(nt, form):
    nr, nz = 5, 7
    print(f"case explicit nt={nt} form={form}", flush=True)
    o, s = make_pair(nt, nr, nz)
    s.set_tuning(explicit_form=form)
    seed_random(o, s, seed=nt)
    o.set_time(0.13)
    s.set_time(0.13)
    substeps(o, s)


# rms error of dq2 against the oracle with the divisions by r and by the last
# diagonal of the theta solve as such: 1.131e-16 and 8.26e-9; bare products with
# rounded inverses 1.200e-16 and 8.93e-9
@pytest.mark.parametrize("precision,nt,nr,nz,bound", [("fp64", 64, 96, 64, 1.15e-16), ("mixed", 16, 24, 40, 8.4e-9)])
def test_plane_form_divides_to_the_last_bit(precision, nt, nr, nz, bound):
    print(f"case plane form accuracy {precision}", flush=True)
    err = []
    for seed in range(3):
        o, s = make_pair(nt, nr, nz, precision=precision)
        s.set_tuning(explicit_form=0)
        seed_random(o, s, seed=seed)
        o.set_time(0.13)
        s.set_time(0.13)
        for p in ["ucoeff", "coesys", "hdnbc", "hdnl1", "hdnl2", "hdnl3", "step"]:
            assert o.phase(p, 1) == 0
        for p in ["hdnbc", "explicit", "adi"]:
            s.phase(p, 1)
        a, b = (x[:, 1 : nr + 1, 1 : nz + 1] for x in (s.download("dq2"), o.field("dq2")))
        err.append(np.sqrt(np.mean((a - b) ** 2) / np.mean(b**2)))
    assert np.mean(err) <= bound, err


# r segments 16 and 24, z segments 16, 24 and 40; the last two run one by one
@pytest.mark.parametrize("nt,nr,nz", [(5, 15, 16), (7, 16, 15), (9, 255, 30), (3, 17, 256), (8, 264, 31), (5, 271, 256),
                                      (4, 12, 520), (3, 271, 512), (3, 300, 20), (4, 9, 700)])
def test_sweeps_of_all_segments_match_oracle(nt, nr, nz):
    print(f"case sweeps {nt}x{nr}x{nz}", flush=True)
    o, s = make_pair(nt, nr, nz, slip=0.25)
    seed_random(o, s, seed=nr + nz)
    o.set_time(0.13)
    s.set_time(0.13)
    substeps(o, s)


@pytest.mark.parametrize("nt,nr,nz,M", [(33, 16, 200, 0), (16, 32, 300, 0), (8, 16, 513, 0), (16, 32, 60, 32),
                                        (16, 32, 60, 48)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_whole_steps_grouped_and_single(nt, nr, nz, M, precision):
    """hdnbc rides in the grouped sweeps of a whole step (M = 0: the default
    segments) and runs by itself beside single ones; 5 steps of a ring, FP64
    to the 1e-10 of the 100-step test, mixed to its 1e-6."""
    print(f"case whole step {nt}x{nr}x{nz} M={M} {precision}", flush=True)
    rmax, zmax = 4.0, 12.0
    q1, q2, q3 = vring_amd.ring_initial_condition(nt, nr, nz, rmax, zmax, [(1.0, 3.0, 0.4, 1.0)])
    dt = vring_amd.cfl_dt(nt, nr, nz, rmax, zmax, q1, q2, q3, cfl=0.3, ujet=1.0)
    o, s = make_pair(nt, nr, nz, rmax, zmax, Re=500.0, dt=dt, precision=precision)
    if M:
        s.set_tuning(M=(M,) * 6)
    seed_fields(o, s, q1, q2, q3)
    for _ in range(5):
        assert o.rk3_step() == 0
    s.step(5)
    vscale = max(np.abs(o.field("q2")).max(), np.abs(o.field("q3")).max())
    compare(o, s, ["q1", "q2", "q3"], 1e-10 if precision == "fp64" else 1e-6, scale=vscale)


# a chosen z tile width runs the mixed path's FP64 low modes by themselves
@pytest.mark.parametrize("nt,nr,nz", [(8, 15, 16), (32, 64, 128), (16, 17, 64), (9, 33, 40), (4, 256, 33), (64, 40, 512),
                                      (16, 12, 1024), (8, 257, 32)])
def test_mixed_modes_in_one_launch_and_apart_agree(nt, nr, nz):
    """Bit for bit: the same sums, whichever launch they are in."""
    print(f"case mixed modes {nt}x{nr}x{nz}", flush=True)
    q1, q2, q3 = vring_amd.ring_initial_condition(nt, nr, nz, 4.0, 12.0, [(1.0, 3.0, 0.4, 1.0)])
    dt = vring_amd.cfl_dt(nt, nr, nz, 4.0, 12.0, q1, q2, q3, cfl=0.3, ujet=1.0)
    got = []
    for lines in (0, 16):
        s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 500.0, dt, precision="mixed")
        s.set_tuning(dct_lines=lines)
        for n, a in (("q1", q1), ("q2", q2), ("q3", q3)):
            s.upload(n, a)
        s.step(3)
        got.append([s.download(n) for n in ("q1", "q2", "q3", "pres")])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_kernel_timer_times_the_kernels_alone():
    """Nine r and z sweeps, three outlet rows and six radial solves a step, on
    a grid whose untimed steps group them."""
    s = vring_amd.Solver(16, 24, 32, 4.0, 12.0, 500.0, 0.01, precision="mixed")
    s.step(1)
    s.enable_ktimer(True)
    s.step(2)
    n = {k: cnt for k, (_, cnt) in s.kernel_times().items()}
    assert (n["line_r"], n["line_z"], n["hdnbc"], n["radial"]) == (18, 18, 6, 12), n
