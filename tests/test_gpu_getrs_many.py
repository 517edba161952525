"""PDGETRS with more right-hand sides than one launch takes (blocked solves), at
the edges of its 256-row blocks, 32-row steps and 16-column strips.

L and U have off-diagonal entries of at most 1 / (2 sqrt(n)), U a diagonal of 1 .. 2
(condition numbers below 10):
X against numpy's FP64 solves within 1e-12 of max |x|, a thousand times the
rounding of sums of this length.  The rows between n and the leading dimension
of A and of B hold NaN.
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
@pytest.mark.parametrize("n,nrhs", [(1, 17), (31, 18), (33, 33), (255, 17), (256, 40), (257, 31),
                                    (300, 64), (513, 100), (1000, 1030)])
def test_many_right_hand_sides(dev, n, nrhs, trans):
    rng = np.random.default_rng(n + nrhs)
    low = np.tril(rng.uniform(-0.5, 0.5, (n, n)), -1) / np.sqrt(n)
    up = np.triu(rng.uniform(-0.5, 0.5, (n, n)), 1) / np.sqrt(n) + np.diag(rng.uniform(1, 2, n))
    ipiv = np.array([rng.integers(i, n) for i in range(n)], dtype=np.int32) + 1
    b = rng.standard_normal((n, nrhs))

    a = (np.eye(n) + low) @ up  # P A = L U: undo the interchanges
    for i in reversed(range(n)):
        a[[i, ipiv[i] - 1]] = a[[ipiv[i] - 1, i]]
    ref = np.linalg.solve(a if trans == "N" else a.T, b)

    lda, ldb = n + 1, n + 2
    fa = np.full((n, lda), np.nan)
    fa[:, :n] = (low + up).T
    fb = np.full((nrhs, ldb), np.nan)
    fb[:, :n] = b.T
    da, db, dp = (torch.from_numpy(v).cuda() for v in (fa, fb, ipiv))
    print(f"[gpu] getrs {trans} n={n} nrhs={nrhs}", flush=True)
    dev.dgetrs_trans(trans, n, nrhs, da, lda, dp, db, ldb)
    got = db.cpu().numpy()
    assert np.isnan(got[:, n:]).all()
    assert np.abs(got[:, :n].T - ref).max() <= 1e-12 * np.abs(ref).max()
