"""Which pivot the last block's LU takes beside NaNs, at every size class of its
kernels (four, eight and twelve wavefronts, and in place beyond 192 columns): a
NaN is no candidate, so a column of one NaN and zeros has a zero pivot and the
factorization fails; a column of nothing but NaNs keeps its diagonal and fails
nothing."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nc", [5, 64, 65, 128, 129, 192, 193])
def test_nan_beside_zeros(Nc):
    print(f"case Nc={Nc}", flush=True)
    s = systems.gaussian_system(1, 2, Nc - 4, Nc - 4, 0, 0, shift=4.0, seed=Nc)
    s["D"][0, :, 0] = 0.0        # the last block's column 0: D_0 over H
    s["H"][:, 0] = 0.0
    for row in (0, 1, Nc - 1):
        t = dict(s, D=s["D"].copy(), H=s["H"].copy())
        if row < 2:
            t["D"][0, row, 0] = np.nan
        else:
            t["H"][row - 2, 0] = np.nan
        g = BorderedCR(np.float64)
        g.load_system(t)
        g.select("LU", "LU", "NONE")
        assert not g.factorize(), row
    t["D"][0, :, 0] = np.nan
    t["H"][:, 0] = np.nan
    g.load_system(t)
    assert g.factorize(), g.last_error()
