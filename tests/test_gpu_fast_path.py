"""fast_path() says whether register-resident LU kernels eliminated the pairs:
with N = 1 there are none to eliminate, whatever the block size."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import BorderedCR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 8, 16, 17, 48])
def test_fast_path_needs_a_pair(n, dtype):
    for N, fast in ((1, False), (2, True), (3, True), (40, True)):
        print(f"case n={n} N={N} {np.dtype(dtype).name}", flush=True)
        g = BorderedCR(dtype)
        g.load_system(systems.gaussian_system(N, n, 1, 1, 2, 2, shift=4.0, seed=N))
        assert g.factorize(), g.last_error()
        assert g.fast_path() == fast
