"""Batched solves at the edges of their 64-row blocks, 16-row triangles and tiles and
1 .. 16 right-hand sides, shuffled rows, padded leading dimensions holding NaN.

A is uniform in [-1, 1) with n added on the diagonal, rows shuffled: condition number
below 10, X within 1e-12 (FP32: times 2^29) of max |x| of numpy's FP64 solution, some
thousand times the rounding of sums of this length.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dev():
    from scalapack_amd.device import Handle
    h = Handle()
    yield h
    h.close()


def _solve(dev, prec, mats, rhs):
    dt = np.float64 if prec == "fp64" else np.float32
    ns, nr = [a.shape[0] for a in mats], [b.shape[1] for b in rhs]
    fa, fb = [], []
    for a, b in zip(mats, rhs):
        n = a.shape[0]
        pa, pb = np.full((n, n + 1), np.nan, dt), np.full((b.shape[1] + 1, n + 3), np.nan, dt)
        pa[:, :n], pb[:-1, :n] = a.T, b.T
        fa.append(torch.from_numpy(pa).cuda())
        fb.append(torch.from_numpy(pb).cuda())
    ps = [torch.zeros(n, dtype=torch.int32, device="cuda") for n in ns]
    ptr = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64).cuda()  # noqa: E731
    info = torch.full((len(ns),), -7, dtype=torch.int32, device="cuda")
    dev.gesv_batched(prec, ns, nr, ptr(fa), [n + 1 for n in ns], ptr(ps), ptr(fb),
                     [n + 3 for n in ns], info)
    assert (info.cpu().numpy() == 0).all()
    out = []
    for n, r, b in zip(ns, nr, fb):
        got = b.cpu().numpy()
        assert np.isnan(got[:, n:]).all() and np.isnan(got[r]).all()
        out.append(got[:r, :n].T)
    return out


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nrhs", [1, 3, 4, 5, 16])
def test_edges(dev, nrhs, prec):
    rng = np.random.default_rng(nrhs)
    ns = [1, 2, 15, 16, 17, 48, 63, 64, 65, 80, 127, 128, 129, 500, 512, 513, 1023, 1024]
    mats = [(rng.uniform(-1, 1, (n, n)) + n * np.eye(n))[rng.permutation(n)] for n in ns]
    rhs = [rng.standard_normal((n, nrhs)) for n in ns]
    if prec == "fp32":
        mats, rhs = [a.astype(np.float32).astype(float) for a in mats], \
                    [b.astype(np.float32).astype(float) for b in rhs]
    print(f"[gpu] batched solve {prec} nrhs={nrhs}", flush=True)
    tol = 1e-12 * (1 if prec == "fp64" else 2.0 ** 29)
    for n, a, b, x in zip(ns, mats, rhs, _solve(dev, prec, mats, rhs)):
        ref = np.linalg.solve(a, b)
        assert np.abs(x - ref).max() <= tol * np.abs(ref).max(), n


def test_quotients_without_a_reciprocal(dev):
    """Pivots whose reciprocal overflows, and quotients that overflow."""
    mats = [np.array([[1e-310]]), np.array([[1e-310]]), np.array([[2.0, 1.0], [0.0, 4e-320]])]
    rhs = [np.array([[3e-310]]), np.array([[1.0]]), np.array([[3.0], [4e-320]])]
    x = _solve(dev, "fp64", mats, rhs)
    assert x[0][0, 0] == rhs[0][0, 0] / mats[0][0, 0]
    assert np.isposinf(x[1][0, 0])
    np.testing.assert_array_equal(x[2], [[1.0], [1.0]])
