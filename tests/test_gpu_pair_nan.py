"""Which pivot the register LU pair kernel (n <= 16) takes beside NaNs: a NaN is
behind every number, so a column of one NaN and zeros has a zero pivot and the
factorization fails.  For every register configuration, in the fused launch, in
a launch per level and in a batch."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import Batch, BorderedCR, DeviceArray

pytestmark = pytest.mark.gpu


def nan_beside_zeros(N, n, r, pair, row, col, seed):
    """The T panel [E_{pair - 1}; D_pair] of a pair of the first level: column
    `col` holds zeros and, at panel row `row`, one NaN."""
    s = systems.gaussian_system(N, n, 1, 1, r, r, shift=4.0, seed=seed)
    s["E"][pair - 1, :, col] = 0.0
    s["D"][pair, :, col] = 0.0
    (s["E"][pair - 1] if row < n else s["D"][pair])[row % n, col] = np.nan
    return s


@pytest.mark.parametrize("n,r", [(1, 0), (4, 4), (5, 2), (8, 8), (12, 4), (16, 8)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_nan_beside_zeros(n, r, dtype):
    for N, pair in ((2, 1), (700, 33), (9000, 4099)):
        for row, col in ((1, 0), (n, 0), (2 * n - 1, n - 1)):
            print(f"case n={n} r={r} N={N} row={row} col={col} {np.dtype(dtype).name}", flush=True)
            s = nan_beside_zeros(N, n, r, pair, row, col, seed=n + N)
            for timing in (False, True):
                g = BorderedCR(dtype)
                g.set_timing(timing)
                g.load_system(s)
                g.select("LU", "LU", "NONE")
                assert not g.factorize()


def test_nan_beside_zeros_in_a_batch():
    bt = Batch(mixed=False)
    bt.plan(np.asarray([(40, 3, 1, 1, 2, 2, 0), (40, 6, 1, 1, 2, 2, 0), (40, 13, 1, 1, 2, 2, 0)] * 2, np.int32))
    bt.generate(seed=5, shift=4.0)
    for s, n in ((3, 3), (4, 6), (5, 13)):
        print(f"case batch n={n}", flush=True)
        bt.load_system(s, nan_beside_zeros(40, n, 2, 3, n + 1, 0, seed=n))
    X = DeviceArray(bt.size("x"))
    assert bt.solve(DeviceArray.from_host(np.ones(bt.size("x"))), X, max_iter=2, graph=False) == 2
    assert list(bt.report()["status"] & 1) == [0, 0, 0, 1, 1, 1]   # bit 0: a zero pivot
