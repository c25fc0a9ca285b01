"""Both sides of the lines at which a pair launch changes its kernel by the number
of pairs: the right-hand kernel's waves (256 pairs), the FP32 panel's waves (1024
pairs, n > 32), the unrolled form of the small register kernel (1024 workgroups),
and the fused levels of FP32 objects against a launch per level.

The first level's panels go through the same operations in the same order in
every LU kernel, so T and the pivots are compared bit for bit; D, E, B and C of the
first level's pairs differ in rounding only (1e-12 relative to the largest entry
in FP64, 1e-4 in FP32).  QR panels against the oracle, 1e-11."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR

pytestmark = pytest.mark.gpu


def factored(s, dtype, variant=0, timing=False, method="LU"):
    g = BorderedCR(dtype)
    g.load_system(s)
    g.select(method, "LU", "NONE")
    g.set_pair_kernel(variant)
    g.set_timing(timing)
    assert g.factorize(), g.last_error()
    return g, g.factors()


def same_first_level(fa, fb, s, dtype):
    N, n, nr, nx = s["N"], s["n"], s["nr"], s["nx"]
    ta, tb = (f["T"].reshape(N, -1)[1::2, :2 * n * n] for f in (fa, fb))
    assert np.array_equal(ta, tb)
    assert np.array_equal(fa["perm"].reshape(N, n)[1::2], fb["perm"].reshape(N, n)[1::2])
    rel = 1e-4 if dtype == np.float32 else 1e-12
    for k, w in (("D", n * n), ("E", n * n), ("B", n * nx), ("C", nr * n)):
        if w:
            a, b = (f[k][:N * w].reshape(N, w)[1::2] for f in (fa, fb))
            assert np.abs(a - b).max() <= rel * max(1.0, np.abs(b).max()), k


LINES = [(np.float64, n, N) for n in (17, 32, 33, 48, 49, 64) for N in (513, 515)]
LINES += [(np.float32, n, N) for n in (17, 32, 33, 48, 49, 64) for N in (513, 515)]
LINES += [(np.float32, n, N) for n in (33, 48, 49, 64) for N in (2049, 2051)]


@pytest.mark.parametrize("dtype,n,N", LINES)
def test_lu_pairs(dtype, n, N):
    for nr, nx in ((0, 0), (1, 16), (8, 3)):
        print(f"case n={n} N={N} nr={nr} nx={nx} {np.dtype(dtype).name}", flush=True)
        qr = max(0, nx - nr) + 2
        s = systems.gaussian_system(N, n, qr, qr + nr - nx, nr, nx, shift=4.0, seed=n)
        _, fa = factored(s, dtype)
        _, fb = factored(s, dtype, variant=4)
        same_first_level(fa, fb, s, dtype)


@pytest.mark.parametrize("method", ["QR", "QRP"])
@pytest.mark.parametrize("n", [17, 32, 33, 48])
def test_qr_pairs(oracle_mod, n, method):
    for N, nr, nx in ((513, 8, 3), (515, 1, 16)):
        print(f"case {method} n={n} N={N} nr={nr} nx={nx}", flush=True)
        qr = max(0, nx - nr) + 2
        s = systems.gaussian_system(N, n, qr, qr + nr - nx, nr, nx, shift=3.0 * np.sqrt(n), seed=n)
        o = oracle_mod.OracleBorderedCR(np.float64)
        o.allocate(N, n, qr, qr + nr - nx, nr, nx)
        o.load(s)
        o.select(method, "LU")
        assert o.factorize(), o.last_error()
        g, f = factored(s, np.float64, method=method)
        oi = o.internals()
        for k, w in (("T", 2 * n * n + n), ("D", n * n), ("E", n * n)):
            a, b = (v.ravel()[:N * w].reshape(N, w)[1::2] for v in (f[k], oi[k]))
            assert np.abs(a - b).max() <= 1e-11 * max(1.0, np.abs(b).max()), k
        x = np.random.default_rng(3).standard_normal(systems.dims(s)[1])
        b = systems.mv(s, x)
        ok, y = g.solve(b)
        assert ok and np.linalg.norm(systems.mv(s, y) - b) <= 1e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,r,N", [(n, r, N) for n, rs, Ns in ((4, (0, 4), (16369, 16385)), (8, (4, 8), (8185, 8193)),
                                                               (13, (2,), (4093, 4097)), (16, (4, 8), (4093, 4097)))
                                   for r in rs for N in Ns])
def test_small_pairs(n, r, N, dtype):
    print(f"case n={n} r={r} N={N} {np.dtype(dtype).name}", flush=True)
    s = systems.gaussian_system(N, n, 2, 2, r, r, shift=4.0, seed=n)
    _, fa = factored(s, dtype)
    _, fb = factored(s, dtype, variant=4)
    same_first_level(fa, fb, s, dtype)


@pytest.mark.parametrize("n,r", [(1, 1), (4, 0), (4, 4), (3, 8), (5, 2), (8, 4), (8, 5), (9, 2), (16, 4), (16, 8)])
def test_fused_levels_fp32(n, r):
    for N in (1, 2, 3, 33, 65, 260, 517, 2050):
        print(f"case fp32 n={n} r={r} N={N}", flush=True)
        s = systems.gaussian_system(N, n, n // 2, n // 2, r, r, shift=4.0, seed=100 * n + N)
        g, f = factored(s, np.float32)
        t, ft = factored(s, np.float32, timing=True)   # every level a launch of its own
        if N > 1:
            for k in ("T", "D", "E", "B"):
                a, b = ((v[k].reshape(N, -1)[1:, :2 * n * n] if k == "T" else v[k]) for v in (f, ft))
                assert np.array_equal(a, b), k
        if n * N >= 2500:     # (no dense condition number)
            continue
        rhs = np.random.default_rng(N).standard_normal(systems.dims(s)[0]).astype(np.float32)
        ok, x = g.solve(rhs)
        ok2, y = t.solve(rhs)
        # only the order of the boundary sums differs
        lim = 50 * np.finfo(np.float32).eps * np.linalg.cond(systems.dense(s))
        assert ok and ok2 and np.abs(x - y).max() <= lim * max(1.0, np.abs(y).max())
