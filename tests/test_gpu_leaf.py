"""The panel leaf (PDGETF2 on at most 32 columns) at the edges of its layouts.

The matrices have at most one +1 and one -1 per row, columns scaled by powers
of two: every Schur complement of such a matrix holds only 0 and +-1 (times the
scales), so the elimination is exact in any order, every pivot search ties, and
columns without a pivot occur.  Factors, IPIV and INFO therefore have to equal a
plain numpy elimination exactly (first maximum, reciprocal scaling, a zero pivot
recorded and skipped: SRC/pdgetf2.f:206-237); NaN entries must stay where that
elimination puts them.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dev():
    from scalapack_amd.device import Handle
    h = Handle(nb=64)
    yield h
    h.close()


def incidence(m, n, seed, nans=0):
    rng = np.random.default_rng(seed)
    a = np.zeros((m, n))
    rows = np.arange(m)
    a[rows, rng.integers(0, n, m)] = 1.0
    second = rng.integers(0, 2 * n, m)  # half of the rows have one entry only
    on = (second < n) & (a[rows, np.minimum(second, n - 1)] == 0)
    a[rows[on], second[on]] = -1.0
    a *= 2.0 ** rng.integers(-3, 4, n)
    for _ in range(nans):
        a[rng.integers(0, m), rng.integers(0, n)] = np.nan
    return a


def eliminate(a):
    """(factors, 0-based pivots, INFO) of the unblocked elimination."""
    a, (m, n) = a.copy(), a.shape
    piv, info = np.arange(min(m, n)), 0
    with np.errstate(invalid="ignore"):
        for j in range(min(m, n)):
            mag = np.abs(a[j:, j])
            mag = np.where(np.isnan(mag), -1.0, mag)
            p = j + int(np.argmax(mag))
            if mag[p - j] > 0:
                piv[j] = p
                a[[j, p]] = a[[p, j]]
                a[j + 1:, j] *= 1.0 / a[j, j]
            elif info == 0:
                info = j + 1
            a[j + 1:, j + 1:] -= np.outer(a[j + 1:, j], a[j, j + 1:])
    return a, piv, info


def check(dev, a):
    m, n = a.shape
    lda = m + 3
    buf = np.full((n, lda), 7.0)
    buf[:, :m] = a.T
    t = torch.from_numpy(buf).cuda()
    ipiv = torch.zeros(min(m, n), dtype=torch.int32, device="cuda")
    print(f"[gpu] leaf m={m} n={n}", flush=True)
    info = dev.dgetrf(m, n, t, lda, ipiv)
    lu, piv, want = eliminate(a)
    got = t.cpu().numpy()
    assert info == want
    assert np.array_equal(ipiv.cpu().numpy() - 1, piv)
    assert np.array_equal(got[:, :m].T, lu, equal_nan=True)
    assert (got[:, m:] == 7.0).all(), "rows below the matrix were written"


# one workgroup of 1 .. 8 waves (4 or 8 rows a quad), several workgroups, the
# taller ones with 8 rows a quad; widths of every register count and remainder
@pytest.mark.parametrize("m", [1, 5, 16, 63, 65, 128, 447, 512, 513, 1023, 1025, 2049, 16385, 33000])
@pytest.mark.parametrize("w", [1, 4, 7, 8, 9, 16, 19, 31, 32])
def test_leaf_exact(dev, m, w):
    check(dev, incidence(m, min(w, m), seed=100 * w + m))


@pytest.mark.parametrize("m,n", [(90, 64), (700, 80), (1300, 150), (150, 150), (70, 200)])
def test_leaf_interchanges_reach_the_block_column(dev, m, n):
    check(dev, incidence(m, n, seed=m + n))


@pytest.mark.parametrize("m", [40, 600, 1500])
def test_leaf_nan(dev, m):
    check(dev, incidence(m, 32, seed=m, nans=3))
