"""Shapes whose LDS arrays come out at exactly the limit of a workgroup
(163840 bytes), one below and one beyond: the last solve's block and columns
(Nc = 128 with 16 columns; Nc = 640 the columns alone), a whole pair panel
(n = 32, nx = 224 in FP64) and the back substitution of QR / QRP pairs in a
batch (n = 64, nx = 51: D, E, U, B and 16 columns).  A drawn solution x,
b = A x: |x' - x| <= 50 eps cond relative to the largest entry."""
import numpy as np
import pytest

from alglin_amd import systems
from alglin_amd.bcr import AlglinError, Batch, BorderedCR, DeviceArray

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def drawn(s, m):
    x = np.random.default_rng(7).standard_normal((systems.dims(s)[1], m))
    return x, np.stack([systems.mv(s, x[:, q]) for q in range(m)], 1)


def close(s, y, x):
    return np.abs(y - x).max() <= 50 * EPS * np.linalg.cond(systems.dense(s)) * max(1.0, np.abs(x).max())


@pytest.mark.parametrize("last,last2", [("LUPQ", "NONE"), ("QR", "NONE"), ("QRP", "NONE"), ("LU", "SVD")])
@pytest.mark.parametrize("Nc", [127, 128, 129])
def test_last_solve_block_and_columns(Nc, last, last2):
    n, r, N = 4, 1, 3
    print(f"case Nc={Nc} {last}/{last2}", flush=True)
    s = systems.gaussian_system(N, n, Nc - 2 * n - r, Nc - 2 * n - r, r, r, shift=4.0, seed=Nc)
    x, B = drawn(s, 17)
    g = BorderedCR(np.float64)
    g.load_system(s)
    g.select("LU", last, last2)
    assert g.factorize(), g.last_error()
    ok, X = g.solve_n(B)
    assert ok and close(s, X, x)


@pytest.mark.parametrize("Nc,fits", [(639, True), (640, False), (641, False)])
def test_last_solve_columns(Nc, fits):
    n, r, N = 4, 1, 2
    print(f"case Nc={Nc} LU", flush=True)
    s = systems.gaussian_system(N, n, Nc - 2 * n - r, Nc - 2 * n - r, r, r, shift=4.0, seed=Nc)
    x, B = drawn(s, 2)
    g = BorderedCR(np.float64)
    g.load_system(s)
    g.select("LU", "LU", "NONE")
    assert g.factorize(), g.last_error()
    ok, X = g.solve_n(B)
    assert ok == fits
    if fits:
        assert close(s, X, x)
    else:
        assert "last solve" in g.last_error()
    # a batch of it takes the same arrays
    bt = Batch(mixed=False)
    bt.plan([(N, n, Nc - 2 * n - r, Nc - 2 * n - r, r, r, 0)])
    bt.load_system(0, s)
    Xd = DeviceArray(bt.size("x"))
    b = np.zeros(bt.size("x"))
    b[:B.shape[0]] = B[:, 0]
    if fits:
        bt.solve(DeviceArray.from_host(b), Xd, max_iter=0, graph=False)
        assert close(s, Xd.to_host()[:x.shape[0]], x[:, 0])
    else:
        with pytest.raises(AlglinError):
            bt.solve(DeviceArray.from_host(b), Xd, max_iter=0, graph=False)


@pytest.mark.parametrize("nx,fits", [(223, True), (224, False), (225, False)])
def test_pair_panel(nx, fits):
    """Beyond the limit a single system's panels go through global scratch;
    a batch, which has none, refuses the plan."""
    N, n = 5, 32
    print(f"case panel n={n} nx={nx}", flush=True)
    s = systems.gaussian_system(N, n, nx, 0, 0, nx, shift=4.0, seed=nx)
    x, B = drawn(s, 3)
    g = BorderedCR(np.float64)
    g.load_system(s)
    assert g.factorize(), g.last_error()
    ok, X = g.solve_n(B)
    assert ok and close(s, X, x)
    bt = Batch(mixed=False)
    dims = [(N, n, nx, 0, 0, nx, 0)]
    if not fits:
        with pytest.raises(AlglinError):
            bt.plan(dims)
        return
    bt.plan(dims)
    bt.load_system(0, s)
    Xd = DeviceArray(bt.size("x"))
    b = np.zeros(bt.size("x"))
    b[:B.shape[0]] = B[:, 0]
    bt.solve(DeviceArray.from_host(b), Xd, max_iter=0, graph=False)
    assert close(s, Xd.to_host()[:x.shape[0]], x[:, 0])


@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("n,nx", [(64, 50), (64, 51), (64, 90), (48, 163), (48, 164), (33, 200)])
def test_batched_qr_back_substitution(n, nx, method):
    print(f"case back substitution n={n} nx={nx} method={method}", flush=True)
    N, nr = 6, 2
    s = systems.gaussian_system(N, n, nx - nr, 0, nr, nx, shift=3.0 * np.sqrt(n), seed=nx)
    x, B = drawn(s, 1)
    bt = Batch(mixed=False)
    bt.plan([(N, n, nx - nr, 0, nr, nx, method), (3, 5, 1, 1, 1, 1, method)])
    bt.generate(seed=1, shift=4.0)
    bt.load_system(0, s)
    Xd = DeviceArray(bt.size("x"))
    b = np.zeros(bt.size("x"))
    b[:B.shape[0]] = B[:, 0]
    rc = bt.solve(DeviceArray.from_host(b), Xd, max_iter=0, graph=False)
    assert rc in (0, 2) and close(s, Xd.to_host()[:x.shape[0]], x[:, 0])
