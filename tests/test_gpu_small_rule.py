"""The level from which the fused small-system launch takes over follows the
register configuration of that launch: a block of n = 4 with a border of 8 runs
in the n <= 8 configuration, as n = 5 with the same border does, and so costs no
more than that one.  Medians of 30 factorizations; counted by n alone it took
1.6 times as long."""
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
    a, b = median_time(4, N, 8), median_time(5, N, 8)
    print(f"case N={N}: n = 4 {1e6 * a:.0f} us, n = 5 {1e6 * b:.0f} us", flush=True)
    assert a <= 1.15 * b
