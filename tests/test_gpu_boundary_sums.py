"""The sums of the border partials over all pairs (F and the border unknowns'
right-hand side), at row widths nr nx and nr nrhs on both sides of the reduction
kernel's 128-column line and that do not divide its 256 threads, against the
oracle.  Well-posed systems (condition numbers of a few hundred), FP64 sums of a
few hundred terms: 1e-11 relative to the largest entry."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nx", [(1, 1), (3, 5), (8, 16), (13, 10), (16, 16)])
@pytest.mark.parametrize("N", [2, 17, 400])
def test_border_sums(oracle_mod, N, nr, nx):
    n = 18
    print(f"case N={N} nr={nr} nx={nx}", flush=True)
    q = max(0, nx - nr) + 2
    qx = q + nr - nx
    s = systems.gaussian_system(N, n, q, qx, nr, nx, shift=4.0, seed=N + nr)
    s["C"] /= np.sqrt(N * n)
    s["H"] /= np.sqrt(n)
    rows = np.arange(n + q)
    s["H"][rows, n + rows] += 4.0
    k = np.arange(min(s["F"].shape))
    s["F"][k, k] += 4.0
    o = oracle_mod.OracleBorderedCR(np.float64)
    o.allocate(N, n, q, qx, nr, nx)
    o.load(s)
    assert o.factorize()
    g = BorderedCR(np.float64)
    g.load_system(s)
    assert g.factorize(), g.last_error()
    B = np.random.default_rng(2).standard_normal((systems.dims(s)[0], 20))
    ok, Xo = o.solve_n(B)
    assert ok
    for m in (1, 7, 20):
        ok, X = g.solve_n(B[:, :m])
        assert ok and np.abs(X - Xo[:, :m]).max() <= 1e-11 * np.abs(Xo).max()
