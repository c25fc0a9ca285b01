"""The matrix-core LU pair at the edges of its 16-column blocks and 16-row
tiles (n, n + nr and nx around multiples of 16, no border, the widest border),
against the column-split rank-1 kernel: the T panel, the pivots and C_j U^-1
see the same operations in the same order (the matrix products accumulate as
the chain of fused multiply-adds), so the first level's panels are the same
bits; D, E, B differ in rounding only (1e-12 relative to the largest entry in
FP64, 1e-4 in FP32), and the solution is the oracle's."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR

pytestmark = pytest.mark.gpu


def factored(s, variant, dtype):
    g = BorderedCR(dtype)
    g.load_system(s)
    g.set_pair_kernel(variant)
    assert g.factorize(), g.last_error()
    return g, g.factors()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nr,nx", [(0, 0), (1, 16), (8, 2), (8, 16), (5, 1)])
@pytest.mark.parametrize("n", [15, 16, 17, 24, 31, 32, 33, 40, 47, 48, 49, 56, 63, 64])
def test_panels_equal_the_rank_one_kernel(oracle_mod, n, nr, nx, dtype):
    if n + nr > (48 if n <= 32 else 64 if n <= 48 else 80):
        pytest.skip("beyond the matrix-core pair's shapes")
    N = 11
    qr = max(0, nx - nr) + 2
    qx = qr + nr - nx
    print(f"case n={n} nr={nr} nx={nx} {np.dtype(dtype).name}", flush=True)
    s = systems.gaussian_system(N, n, qr, qx, nr, nx, shift=4.0, seed=n + nr)
    a, fa = factored(s, 5, dtype)
    b, fb = factored(s, 4, dtype)
    ta, tb = (f["T"].reshape(N, -1)[1::2, :2 * n * n] for f in (fa, fb))
    assert np.array_equal(ta, tb)
    assert np.array_equal(fa["perm"].reshape(N, n)[1::2], fb["perm"].reshape(N, n)[1::2])
    rel = 1e-4 if dtype == np.float32 else 1e-12
    for k in ("D", "E", "B", "C"):
        if fb[k].size:
            assert np.abs(fa[k] - fb[k]).max() <= rel * max(1.0, np.abs(fb[k]).max()), k
    rhs = np.random.default_rng(1).standard_normal(systems.dims(s)[0]).astype(dtype)
    ok, x = a.solve(rhs)
    ok2, y = b.solve(rhs)
    cond = np.linalg.cond(systems.dense(s))
    eps = np.finfo(dtype).eps
    assert ok and ok2 and np.abs(x - y).max() <= 50 * eps * cond * max(1.0, np.abs(y).max())
    assert a.factorize()     # again: no pending border term survives
    ok, z = a.solve(rhs)
    assert ok and np.array_equal(x, z)
