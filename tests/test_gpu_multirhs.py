"""Several right-hand sides on the GPU: the matrix-core sweeps at the edges of
their 16-row and 16-column tiles, against the same system solved one column at
a time (the one-column sweeps, checked against the oracle elsewhere) and
against the oracle.  Both orders of the sums are FP64 with the same factors:
1e-12 relative to the largest entry of a solution of these well-conditioned
systems; FP32 objects 1e4 eps32 (condition numbers of a few hundred)."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR, DeviceArray, packed_blocks

pytestmark = pytest.mark.gpu


def well_posed(N, n, r, seed):
    """Boundary rows with their weight on the last block, border rows scaled
    to quadratures: condition numbers of a few hundred at most."""
    q = n // 4
    s = systems.gaussian_system(N, n, q, q, r, r, shift=4.0, seed=seed)
    s["C"] /= np.sqrt(N * n)
    s["H"] /= np.sqrt(n)
    s["H"][np.arange(n + q), n + np.arange(n + q)] += 4.0
    s["F"][np.arange(r), np.arange(r)] += 4.0
    return s


@pytest.mark.parametrize("method", ["LU", "QR"])
@pytest.mark.parametrize("n", [1, 8, 9, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64])
def test_columns_together_equal_columns_alone(oracle_mod, n, method):
    for N, r in ((1, 1), (2, 0), (7, 3), (130, 8 if n > 8 else 2), (300, 16 if n > 16 else 1)):
        s = well_posed(N, n, r, seed=n + N)
        nrows, ncols = systems.dims(s)
        g = BorderedCR(np.float64)
        g.load_system(s)
        g.select(method, "LU", "NONE")
        assert g.factorize(), g.last_error()
        B = np.random.default_rng(n).standard_normal((nrows, 33))
        one = np.stack([g.solve(B[:, c])[1] for c in range(33)], 1)
        scale = np.abs(one).max()
        for m in (2, 5, 16, 17, 33):
            print(f"case n={n} N={N} r={r} nrhs={m} {method}", flush=True)
            ok, X = g.solve_n(B[:, :m])
            assert ok and np.abs(X - one[:, :m]).max() < 1e-12 * scale
        if N > 1 and method == "LU":
            o = oracle_mod.OracleBorderedCR(np.float64)
            o.allocate(N, n, s["qr"], s["qx"], r, r)
            o.load(s)
            assert o.factorize()
            ok, Xo = o.solve_n(B)
            assert ok and np.abs(one - Xo).max() < 1e-11 * scale


@pytest.mark.parametrize("n", [5, 12, 24, 40, 57])
def test_fp32_mixed_and_leading_dimension(n):
    N, r, m, pad = 70, 2, 6, 5
    s = well_posed(N, n, r, seed=n)
    nrows, ncols = systems.dims(s)
    x = np.random.default_rng(3).standard_normal((ncols, m))
    B = systems.mv(s, x)
    f = BorderedCR(np.float32)
    f.load_system(s)
    assert f.factorize(), f.last_error()
    ok, y = f.solve_n(B.astype(np.float32))
    assert ok and np.abs(y - x).max() < 200 * np.finfo(np.float32).eps * np.abs(x).max() * 50
    # device columns with a leading dimension beyond the rows: the gap stays as it was
    pk = packed_blocks(s)
    dev = {k: DeviceArray.from_host(v) for k, v in pk.items()}
    for mode in ("FP64", "MIXED"):
        g = BorderedCR(np.float64)
        g.allocate(N, n, s["qr"], s["qx"], r, r)
        g.select_precision(mode, 1e-12)
        g.bind_device(dev)
        assert g.factorize_device(), g.last_error()
        ld = nrows + pad
        X = np.full((m, ld), 7.0)
        X[:, :nrows] = B.T
        xd = DeviceArray.from_host(X)
        g.solve_device(xd, m, ld)
        out = xd.to_host().reshape(m, ld)
        assert np.abs(out[:, :ncols].T - x).max() < 1e-10 * np.abs(x).max()
        assert (out[:, nrows:] == 7.0).all()
