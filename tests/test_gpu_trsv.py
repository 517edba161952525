"""PDGETRS with up to 16 right-hand sides (one launch a triangle), at the edges of
its 64-row blocks, 16-row triangles and 1, 4 or 16 columns.

Factors and tolerance as for many right-hand sides: L and U have off-diagonal
entries of at most 1 / (2 sqrt(n)), U a diagonal of 1 .. 2, and X is within 1e-12
of max |x| of numpy's FP64 solves.  Rows between n and the leading dimensions hold
NaN, as do the columns of B after the last right-hand side.
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


@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 130, 449, 1024])
def test_right_hand_sides_to_16(dev, n, trans):
    rng = np.random.default_rng(n)
    low = np.tril(rng.uniform(-0.5, 0.5, (n, n)), -1) / np.sqrt(n)
    up = np.triu(rng.uniform(-0.5, 0.5, (n, n)), 1) / np.sqrt(n) + np.diag(rng.uniform(1, 2, n))
    ipiv = np.array([rng.integers(i, n) for i in range(n)], dtype=np.int32) + 1
    a = (np.eye(n) + low) @ up  # P A = L U: undo the interchanges
    for i in reversed(range(n)):
        a[[i, ipiv[i] - 1]] = a[[ipiv[i] - 1, i]]
    lda, ldb = n + 1, n + 2
    fa = np.full((n, lda), np.nan)
    fa[:, :n] = (low + up).T
    da, dp = torch.from_numpy(fa).cuda(), torch.from_numpy(ipiv).cuda()
    for nrhs in (1, 2, 3, 4, 5, 13, 16):
        b = rng.standard_normal((n, nrhs))
        ref = np.linalg.solve(a if trans == "N" else a.T, b)
        fb = np.full((nrhs + 1, ldb), np.nan)
        fb[:nrhs, :n] = b.T
        db = torch.from_numpy(fb).cuda()
        print(f"[gpu] getrs {trans} n={n} nrhs={nrhs}", flush=True)
        dev.dgetrs_trans(trans, n, nrhs, da, lda, dp, db, ldb)
        got = db.cpu().numpy()
        assert np.isnan(got[:, n:]).all() and np.isnan(got[nrhs]).all()
        assert np.abs(got[:nrhs, :n].T - ref).max() <= 1e-12 * np.abs(ref).max()
