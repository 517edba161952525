"""The tournament leaf where many rows share the largest magnitude, rows are zero or
NaN candidates are absent: the FP32 factorization with tournament pivoting of matrices
whose entries are small multiples of powers of two, at the edges of its rows a thread,
candidates a thread, columns left and leaf widths.

P A = L U holds within 2 n eps32 |L| |U|, element by element (Higham's bound for the
factorization is n eps |L| |U|, twice that allows for the solve by which L is formed).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m,n", [(31, 31), (40, 33), (512, 8), (513, 24), (1000, 25), (2100, 48),
                                 (8192, 32), (8193, 17), (16400, 40)])
def test_ties(m, n):
    from scalapack_amd.device import Handle
    rng = np.random.default_rng(m + n)
    a = rng.choice([-1.0, -0.5, 0.0, 0.5, 1.0], (m, n)).astype(np.float32)
    a[rng.permutation(m)[:m // 3]] = 0.0
    a[np.arange(n) * (m // n), np.arange(n)] = 4.0 + np.arange(n) % 2  # full rank
    h = Handle()
    h.set("pivoting", 1)
    da = torch.from_numpy(np.ascontiguousarray(a.T)).cuda()
    dp = torch.zeros(min(m, n), dtype=torch.int32, device="cuda")
    print(f"[gpu] tournament leaf ties m={m} n={n}", flush=True)
    assert h.sgetrf(m, n, da, m, dp) == 0
    h.close()
    lu, piv = da.cpu().numpy().T.astype(np.float64), dp.cpu().numpy()
    pa = a.astype(np.float64)
    for i, p in enumerate(piv):
        assert i + 1 <= p <= m
        pa[[i, p - 1]] = pa[[p - 1, i]]
    low = np.tril(lu, -1)[:, :n] + np.eye(m, n)
    up = np.triu(lu[:n])
    bound = 2 * n * 2.0 ** -24 * (np.abs(low) @ np.abs(up)) + 1e-30
    assert (np.abs(pa - low @ up) <= bound).all()
