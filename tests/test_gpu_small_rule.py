"""The level from which the fused small-system launches take over.

Factorization: it follows the register configuration of the launch: a block of
n = 4 with a border of 8 runs in the n <= 8 configuration, as n = 5 with the same
border does, and so costs no more than that one.  Medians of 30 factorizations;
counted by n alone it took 1.6 times as long.

Solve: a level takes one round of the workgroup, and less with many border sums
per pair: four columns with a border of 16 against one column with a border of 2
take 3.3 times as long at n = 8, 3.9 at n = 2 and 4; with two rounds for either
3.9 and 4.6 to 4.8, slower than a launch per level.

Another load on the machine can spoil a timing, so the best of three counts; the
ratios above are far enough apart for that."""
import time

import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR, DeviceArray, packed_blocks

pytestmark = pytest.mark.gpu


def median_time(n, N, r):
    g = BorderedCR(np.float64)
    s = systems.gaussian_system(N, n, 1, 1, r, r, shift=4.0, seed=n)
    g.allocate(N, n, 1, 1, r, r)
    g.bind_device({k: DeviceArray.from_host(v) for k, v in packed_blocks(s).items()})
    t = []
    for _ in range(35):
        t0 = time.perf_counter()
        assert g.factorize_device()
        t.append(time.perf_counter() - t0)
    return np.median(t[5:])


@pytest.mark.parametrize("N", [600, 1000])
def test_level_rule_counts_the_border(N):
    ratio = []
    while len(ratio) < 3 and not (ratio and min(ratio) <= 1.15):
        a, b = median_time(4, N, 8), median_time(5, N, 8)
        print(f"case N={N}: n = 4 {1e6 * a:.0f} us, n = 5 {1e6 * b:.0f} us", flush=True)
        ratio.append(a / b)
    assert min(ratio) <= 1.15


def solve_time(n, N, r, m):
    s = systems.gaussian_system(N, n, 1, 1, r, r, shift=4.0, seed=n)
    g = BorderedCR(np.float64)
    g.allocate(N, n, 1, 1, r, r)
    g.bind_device({k: DeviceArray.from_host(v) for k, v in packed_blocks(s).items()})
    assert g.factorize_device()
    L = systems.dims(s)[0]
    X = DeviceArray.from_host(np.random.default_rng(0).standard_normal(L * m))
    t = []
    for _ in range(9):      # 20 solves queued: the GPU's time, not the host's
        g.solve_device(X, m, L)
        t0 = time.perf_counter()
        for _ in range(19):
            g.solve_device(X, m, L, sync=False)
        g.solve_device(X, m, L)
        t.append((time.perf_counter() - t0) / 20)
    return np.median(t[1:])


@pytest.mark.parametrize("n,N,times", [(8, 1000, 3.6), (8, 4000, 3.6), (4, 1000, 4.35), (2, 1000, 4.35)])
def test_solve_level_rule_counts_the_work(n, N, times):
    ratio = []
    while len(ratio) < 3 and not (ratio and min(ratio) <= times):
        a, b = solve_time(n, N, 2, 1), solve_time(n, N, 16, 4)
        print(f"case n={n} N={N}: 1 column {1e6 * a:.0f} us, border of 16 and 4 columns {1e6 * b:.0f} us", flush=True)
        ratio.append(b / a)
    assert min(ratio) <= times
