"""LU classes of a batch whose members lie on both sides of the kernels' block
counts: a launch takes the 16-column blocks of its largest n, and a smaller
member's border rows C_j (panel rows 2n ..) then begin in an earlier 16-row tile
than those of the largest.  Every system against the oracle, without a
refinement sweep: 50 eps cond relative to the largest entry of x."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import Batch, DeviceArray

pytestmark = pytest.mark.gpu


def check(oracle_mod, bt, b, x, eps):
    for s, (N, n, qr, qx, nr, nx, _) in enumerate(bt.dims):
        sysd = bt.system(s)
        nrows, ncols = systems.dims(sysd)
        o = oracle_mod.OracleBorderedCR(np.float64)
        o.allocate(N, n, qr, qx, nr, nx)
        o.load(sysd)
        o.select("LU", "LU")
        assert o.factorize(), o.last_error()
        off = bt.offset("x", s)
        ok, xo = o.solve(b[off:off + nrows])
        assert ok
        err = np.abs(x[off:off + ncols] - xo[:ncols]).max() / max(1.0, np.abs(xo[:ncols]).max())
        assert err <= 50 * eps * np.linalg.cond(systems.dense(sysd)), (s, n, nr, err)


def solved(dims, mixed, max_iter):
    bt = Batch(mixed=mixed)
    bt.plan(np.asarray(dims, np.int32))
    bt.generate(seed=5, shift=4.0)
    b = np.random.default_rng(2).standard_normal(bt.size("x"))
    X = DeviceArray(bt.size("x"))
    rc = bt.solve(DeviceArray.from_host(b), X, tol=1e-12, max_iter=max_iter, graph=False)
    return bt, b, X.to_host(), rc


# (ns of one class; the borders)
CLASSES = [([33, 36, 40, 47, 48, 49, 53, 56, 63, 64], "n64"), ([33, 40, 48], "n48"), ([17, 24, 25, 32], "n32")]


@pytest.mark.parametrize("nr", [0, 1, 2, 5, 8])
@pytest.mark.parametrize("ns", [c[0] for c in CLASSES], ids=[c[1] for c in CLASSES])
def test_border_rows_fp64(oracle_mod, ns, nr):
    print(f"case batch border fp64 ns={ns} nr={nr}", flush=True)
    dims = [(N, n, 3, 3, nr, nr, 0) for n in ns for N in (2, 9)]
    bt, b, x, _ = solved(dims, False, 0)
    check(oracle_mod, bt, b, x, np.finfo(np.float64).eps)


@pytest.mark.parametrize("nr", [1, 3, 8])
def test_border_rows_small_blocks_with_wide_parameters(oracle_mod, nr):
    """n <= 16 with nx > 8 shares the class of the large blocks."""
    print(f"case batch border nx=16 nr={nr}", flush=True)
    dims = [(7, n, 20 - nr, 4, nr, 16, 0) for n in (3, 8, 16, 17, 32, 47)] + [(5, 64, 3, 3, nr, nr, 0)]
    bt, b, x, _ = solved(dims, False, 0)
    check(oracle_mod, bt, b, x, np.finfo(np.float64).eps)


@pytest.mark.parametrize("nr", [1, 8])
def test_border_rows_fp32_factors(oracle_mod, nr):
    print(f"case batch border fp32 nr={nr}", flush=True)
    dims = [(N, n, 3, 3, nr, nr, 0) for n in (33, 40, 47, 48, 49, 56, 64) for N in (2, 9)]
    bt, b, x, _ = solved(dims, True, 0)
    check(oracle_mod, bt, b, x, np.finfo(np.float32).eps)
