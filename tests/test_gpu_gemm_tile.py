"""C -= A B at the edges of the 64 x 64 (n <= 32: 64 x 32) tiles and 16-deep
steps, unaligned leading dimensions included.

Whole-number operands small enough that every sum is exact in FP64: the result
has to be equal, and nothing outside the m x n block may change.
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


def padded(a, ld, fill):
    buf = np.full((a.shape[1], ld), fill)
    buf[:, :a.shape[0]] = a.T
    return torch.from_numpy(buf).cuda()


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (15, 33, 16), (16, 32, 15), (17, 31, 17), (63, 64, 1), (64, 65, 31), (65, 63, 33),
    (128, 1, 64), (1, 128, 48), (129, 40, 100), (640, 32, 32), (700, 513, 20), (1100, 1030, 7)])
@pytest.mark.parametrize("pad", [0, 1, 3])
def test_tile_edges(dev, m, n, k, pad):
    rng = np.random.default_rng(m + 1000 * n + k)
    a, b, c = (rng.integers(-9, 10, s).astype(np.float64) for s in ((m, k), (k, n), (m, n)))
    da, db, dc = padded(a, m + pad, np.nan), padded(b, k + pad, np.nan), padded(c, m + pad, 5.0)
    print(f"[gpu] gemm {m} {n} {k} pad {pad}", flush=True)
    dev.dgemm_sub(m, n, k, da, m + pad, db, k + pad, dc, m + pad)
    got = dc.cpu().numpy()
    assert np.array_equal(got[:, :m].T, c - a @ b)
    assert (got[:, m:] == 5.0).all()
