"""The dense FP64 matrix-core transforms (vrh_dense.hip) against the oracle at
the edges of their tiles: lengths around multiples of 16 and 32, odd and even,
the shortest and longest, line counts that fill no block, and the two tile
widths (32 lines per block from 16384 lines on, up to 320 z points)."""
import numpy as np
import pytest

from gpu_common import make_pair

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
