"""The dense FP64 matrix-core transforms (vrh_dense.hip) against the oracle at
the edges of their tiles: lengths around multiples of 16 and 32, odd and even,
the shortest and longest, line counts that fill no block, and the two tile
widths (32 lines per block from 8192 lines on, up to 320 z points)."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from gpu_common import make_pair
from oracle_lib import Oracle

import vring_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,nr,nz", [(3, 4, 5), (5, 7, 17), (6, 9, 31), (7, 5, 33), (31, 6, 63), (33, 4, 65), (34, 5, 6),
                                      (254, 5, 12), (255, 4, 9), (16, 6, 48), (12, 9, 64), (4, 5, 1150), (33, 500, 20)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_poisson_of_other_lengths_matches_oracle(nt, nr, nz, precision):
    """FP64 to the 1e-11 of the other pressure tests; mixed to its radial
    solves' FP32 rounding (2e-5, as test_gpu_parity)."""
    print(f"case dense poisson {nt}x{nr}x{nz} {precision}", flush=True)
    o, s = make_pair(nt, nr, nz, precision=precision)
    rhs = np.random.default_rng(3).standard_normal((nt, nr, nz))
    ref = o.poisson(rhs)
    got = s.poisson(rhs)
    tol = 1e-11 if precision == "fp64" else 2e-5
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()


# 8192 and more lines, where a block takes two tiles of 16 up to 320 points (more
# than 64 KB of LDS beyond 256) and one beyond
WIDE = [(64, 128, 300), (64, 128, 320), (64, 128, 321)]


@pytest.fixture(scope="module")
def wide_references():
    """The oracle's solutions (its direct z sums take 25 s each), side by side."""
    def solve(g):
        o = Oracle(*g, 4.0, 12.0, 1000.0, 0.01, 0.0, wvnex=1)
        return o.poisson(np.random.default_rng(3).standard_normal(g))
    with ThreadPoolExecutor(len(WIDE)) as ex:
        return dict(zip(WIDE, ex.map(solve, WIDE)))


@pytest.mark.parametrize("grid", WIDE)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_poisson_with_wide_tiles_matches_oracle(wide_references, grid, precision):
    print(f"case dense poisson {grid} {precision}", flush=True)
    s = vring_amd.Solver(*grid, 4.0, 12.0, 1000.0, 0.01, precision=precision)
    ref = wide_references[grid]
    got = s.poisson(np.random.default_rng(3).standard_normal(grid))
    tol = 1e-11 if precision == "fp64" else 2e-5
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()
