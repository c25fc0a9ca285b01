"""Several right-hand sides of QR and QRP systems, four columns per pass of the
streamed forward sweep: remainders of a pass, block sizes within and beyond one
chunk of reflectors (16).  And a pass must cost little beside the launches: 64
columns take at most five times what four take (n = 1, N = 3000: 4.1 times; 5.9
with each column's loads and the reflectors waited for in every pass)."""
import time

import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR, DeviceArray, packed_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["QR", "QRP"])
@pytest.mark.parametrize("n", [1, 2, 8, 15, 16, 17, 32, 33, 64])
def test_columns(n, method):
    N = 6
    s = systems.gaussian_system(N, n, 1, 1, 2, 2, shift=3.0 * np.sqrt(n), seed=n)
    x = np.random.default_rng(n).standard_normal((systems.dims(s)[1], 33))
    B = np.stack([systems.mv(s, x[:, q]) for q in range(33)], 1)
    g = BorderedCR(np.float64)
    g.load_system(s)
    g.select(method, "LU", "NONE")
    assert g.factorize(), g.last_error()
    lim = 50 * np.finfo(np.float64).eps * np.linalg.cond(systems.dense(s))
    for m in (1, 2, 3, 4, 5, 16, 17, 33):
        print(f"case {method} n={n} columns={m}", flush=True)
        ok, X = g.solve_n(B[:, :m])
        assert ok and np.abs(X - x[:, :m]).max() <= lim * max(1.0, np.abs(x).max())


def test_many_columns_of_a_small_block():
    N, n = 3000, 1
    s = systems.gaussian_system(N, n, 1, 1, 2, 2, shift=4.0, seed=1)
    g = BorderedCR(np.float64)
    g.allocate(N, n, 1, 1, 2, 2)
    g.bind_device({k: DeviceArray.from_host(v) for k, v in packed_blocks(s).items()})
    g.select("QR", "LU", "NONE")
    assert g.factorize_device()
    L = systems.dims(s)[0]
    X = DeviceArray.from_host(np.random.default_rng(0).standard_normal(L * 64))

    def median(m):
        t = []
        for _ in range(35):
            t0 = time.perf_counter()
            g.solve_device(X, m, L)
            t.append(time.perf_counter() - t0)
        return np.median(t[5:])

    ratio = []
    while len(ratio) < 3 and not (ratio and min(ratio) <= 5):   # another load can spoil a timing
        a, b = median(4), median(64)
        print(f"case 4 columns {1e6 * a:.0f} us, 64 columns {1e6 * b:.0f} us", flush=True)
        ratio.append(b / a)
    assert min(ratio) <= 5
