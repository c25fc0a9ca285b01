"""QR and column-pivoted QR pairs beyond n = 16 (panel in one launch, the
right-hand columns through 16-reflector blocks on the matrix cores in another)
at the edges of the 16-wide blocks, with no border and with the widest: the
factors and the solution against the oracle.  Block reflectors sum in another
order than one reflector at a time; both are backward stable with constants of
a few n, so 1e-11 relative to the largest entry in FP64 for these shifted
Gaussian blocks, and 2e3 eps32 times the last block's growth (taken as 10) in
FP32."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("method", ["QR", "QRP"])
@pytest.mark.parametrize("nr,nx", [(0, 0), (1, 16), (8, 2), (8, 16)])
@pytest.mark.parametrize("n", [16, 17, 24, 31, 32, 33, 40, 47, 48, 49, 63, 64])
def test_split_pairs_match_the_oracle(oracle_mod, n, nr, nx, method, dtype):
    N = 7
    qr = max(0, nx - nr) + 2
    qx = qr + nr - nx
    print(f"case n={n} nr={nr} nx={nx} {method} {np.dtype(dtype).name}", flush=True)
    s = systems.gaussian_system(N, n, qr, qx, nr, nx, shift=3.0 * np.sqrt(n), seed=n + nr)
    o = oracle_mod.OracleBorderedCR(dtype)
    o.allocate(N, n, qr, qx, nr, nx)
    o.load(s)
    o.select(method, "LU")
    assert o.factorize(), o.last_error()
    g = BorderedCR(dtype)
    g.load_system(s)
    g.select(method, "LU", "NONE")
    assert g.factorize(), g.last_error()
    f, oi = g.factors(), o.internals()
    rel = 1e-11 if dtype == np.float64 else 2e4 * np.finfo(np.float32).eps
    for key, skip in (("T", 2 * n * n + n), ("D", n * n), ("E", n * n)):
        if dtype == np.float32 and method == "QRP":
            break   # partial norms may tie to FP32 rounding: another pivot order
        got, ref = f[key].ravel()[skip:], oi[key].ravel()[skip:]
        assert np.abs(got - ref).max() <= rel * max(1.0, np.abs(ref).max()), key
    if nr and dtype == np.float64:
        got, ref = f["C"].ravel()[n * nr:N * n * nr], oi["C"].ravel()[n * nr:N * n * nr]
        assert np.abs(got - ref).max() <= rel * max(1.0, np.abs(ref).max())
    rhs = np.random.default_rng(1).standard_normal(systems.dims(s)[0]).astype(dtype)
    ok, x = g.solve(rhs)
    ok2, y = o.solve_n(rhs[:, None])
    assert ok and ok2
    cond = np.linalg.cond(systems.dense(s))
    assert np.abs(x - y[:, 0]).max() <= 100 * np.finfo(dtype).eps * cond * max(1.0, np.abs(y).max())
    assert g.factorize()     # again: no pending border term survives
    ok, z = g.solve(rhs)
    assert ok and np.array_equal(x, z)
