"""The fused conjugate-gradient kernels at the edges of their cell loops: fewer
cells than a block, more than one and more than eight strides of 64 x 256
threads, slot counts around 8, slots that converge far apart (and leave the
list), and a solve cut short."""
import numpy as np
import pytest

import vring_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nz,slots", [(16, 4, 1), (16, 37, 9), (48, 400, 3), (64, 2100, 2), (32, 64, 8)])
def test_pcg_reaches_the_direct_solution(nr, nz, slots):
    print(f"case pcg {nr}x{nz}x{slots}", flush=True)
    hz = vring_amd.Helmholtz(nr, nz, slots, stretch=1.0)
    hz.set_modes(np.arange(slots, dtype=np.int32) ** 2)
    f = hz.sample(5, 0)
    p, it, rel, ms = hz.solve(f, "pcg", tol=1e-8, maxit=50000)
    assert np.all(it >= 0) and np.all(rel <= 1.05e-8), (it, rel)
    pd = hz.direct(f)
    # residual and solution to the bounds of the other solver comparisons
    assert np.abs(p - pd).max() <= 1e-5 * np.abs(pd).max()
    if it.max() > 3:
        cut = hz.solve(f, "pcg", tol=1e-8, maxit=3)
        assert np.array_equal(cut[1] < 0, it > 3) and np.all(cut[2][it > 3] > 1e-8)
    hz.close()
