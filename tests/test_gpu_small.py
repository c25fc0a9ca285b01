"""Small block sizes (n <= 16) and the last block on the GPU: the pair kernel
and the fused one-workgroup levels at the edges of their groups (n = 1, 4, 5,
8, 9, 16; border widths on either side of the register classes) and of the
level where the fused launch starts, and the register LU / wavefront solve of
the last block at the edges of its row sets.

Tolerances as elsewhere: FP64 against the oracle (same pivots, same order)
1e-11 relative to the largest solution entry; the fused and the separate
launches share their device code, so the factors are the same bits and only
the boundary sums' order differs (1e-13)."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import Batch, BorderedCR, DeviceArray

pytestmark = pytest.mark.gpu


def oracle_solve(oracle_mod, s, B):
    o = oracle_mod.OracleBorderedCR(np.float64)
    o.allocate(s["N"], s["n"], s["qr"], s["qx"], s["nr"], s["nx"])
    o.load(s)
    o.select("LU", "LU")
    assert o.factorize(), o.last_error()
    ok, X = o.solve_n(B)
    assert ok
    return X


def solver(s):
    g = BorderedCR(np.float64)
    g.load_system(s)
    g.select("LU", "LU", "NONE")
    return g


@pytest.mark.parametrize("n,r", [(1, 1), (4, 0), (4, 4), (5, 2), (8, 4), (8, 5), (9, 2), (16, 4), (16, 8)])
def test_small_levels(oracle_mod, n, r):
    # one block, one pair, levels of exactly / one more than one workgroup's rounds
    for N in (1, 2, 3, 32, 33, 65, 129, 260, 517, 2050):
        print(f"case n={n} r={r} N={N}", flush=True)
        s = systems.gaussian_system(N, n, n // 2, n // 2, r, r, shift=4.0, seed=100 * n + N)
        nrows, _ = systems.dims(s)
        B = np.random.default_rng(N).standard_normal((nrows, 5))
        Xo = oracle_solve(oracle_mod, s, B)
        scale = max(1.0, np.abs(Xo).max())
        g = solver(s)
        assert g.factorize(), g.last_error()
        ok, X = g.solve_n(B)
        ok1, x = g.solve(B[:, 0])
        assert ok and ok1
        assert np.abs(X - Xo).max() < 1e-11 * scale
        assert np.abs(x - Xo[:, 0]).max() < 1e-11 * scale
        f = g.factors()
        t = solver(s)
        t.set_timing(True)      # every level a launch of its own
        assert t.factorize(), t.last_error()
        ft = t.factors()
        for k in ("T", "D", "E", "B"):
            m = n * n * 2 if k == "T" else None
            a, b = f[k], ft[k]
            if m:   # the panels of the eliminated blocks (their tails are not written)
                a, b = (v.reshape(N, -1)[1:, :m] for v in (a, b))
            if N > 1:
                assert np.array_equal(a, b), k
        ok, Xt = t.solve_n(B)
        assert ok and np.abs(Xt - X).max() < 1e-13 * scale * max(1.0, np.linalg.norm(B))


def test_small_fp32_and_mixed():
    s = systems.gaussian_system(700, 7, 3, 3, 2, 2, shift=4.0, seed=3)
    nrows, ncols = systems.dims(s)
    x = np.random.default_rng(0).standard_normal(ncols)
    b = systems.mv(s, x)
    cond = 1e4     # bound for these diagonally shifted systems
    g = BorderedCR(np.float32)
    g.load_system(s)
    assert g.factorize(), g.last_error()
    ok, y = g.solve(b.astype(np.float32))
    assert ok and np.abs(y - x).max() < 50 * np.finfo(np.float32).eps * cond
    m = BorderedCR(np.float64)
    m.allocate(*(s[k] for k in ("N", "n", "qr", "qx", "nr", "nx")))
    m.select_precision("MIXED", 1e-12)
    m.load_system(s)
    assert m.factorize(), m.last_error()
    ok, z = m.solve(b)
    assert ok and m.refine_report()["rel_residual"] <= 1e-12


@pytest.mark.parametrize("Nc", [63, 64, 65, 128, 129, 152, 192, 193, 256, 257])
def test_last_block_sizes(oracle_mod, Nc):
    n, r, N = 4, 1, 3
    q = Nc - 2 * n - r
    print(f"case Nc={Nc}", flush=True)
    s = systems.gaussian_system(N, n, q, q, r, r, shift=4.0, seed=Nc)
    nrows, _ = systems.dims(s)
    B = np.random.default_rng(1).standard_normal((nrows, 3))
    Xo = oracle_solve(oracle_mod, s, B)
    scale = max(1.0, np.abs(Xo).max())
    g = solver(s)
    assert g.factorize(), g.last_error()
    ok, X = g.solve_n(B)
    assert ok and np.abs(X - Xo).max() < 1e-11 * scale * max(1.0, np.linalg.cond(systems.dense(s)) / 1e4)
    # the same system twice in a batch
    bt = Batch(mixed=False)
    bt.plan([(N, n, q, q, r, r, 0)] * 2)
    for k in range(2):
        bt.load_system(k, s)
    L = bt.size("x") // 2
    b = np.zeros(2 * L)
    for k in range(2):
        b[k * L:k * L + nrows] = B[:, k]
    Xd = DeviceArray(2 * L)
    bt.solve(DeviceArray.from_host(b), Xd, max_iter=0, graph=False)
    xb = Xd.to_host()
    for k in range(2):
        assert np.abs(xb[k * L:k * L + Xo.shape[0]] - Xo[:, k]).max() < \
            1e-11 * scale * max(1.0, np.linalg.cond(systems.dense(s)) / 1e4)


def test_nan_block_is_not_a_singular_last_block():
    """A NaN in the boundary rows: the factorization reports no zero pivot,
    the solution is not finite."""
    s = systems.gaussian_system(5, 3, 1, 1, 1, 1, shift=4.0, seed=1)
    s["H"][0, 0] = np.nan
    g = solver(s)
    assert g.factorize()
    ok, x = g.solve(np.ones(systems.dims(s)[0]))
    assert ok and not np.isfinite(x).all()
