"""The 1-norm adds each column from its first row to its last, as the reference does:
equal to that sum bit for bit at the edges of its 256-row, 16-column tiles, with NaN
below the matrix, and NaN and infinity carried through.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m,n", [(1, 1), (255, 16), (256, 17), (257, 15), (512, 1), (700, 33), (3, 100)])
def test_one_norm(m, n):
    from scalapack_amd.device import Handle
    h = Handle()
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n)) * 10.0 ** rng.integers(-8, 8, (m, n))
    buf = np.full((n, m + 3), np.nan)
    buf[:, :m] = a.T
    print(f"[gpu] one norm m={m} n={n}", flush=True)
    da = torch.from_numpy(buf).cuda()
    assert h.dlange("1", m, n, da, m + 3) == np.add.accumulate(np.abs(a), axis=0)[-1].max()
    da[n - 1, m - 1] = -np.inf
    assert np.isposinf(h.dlange("1", m, n, da, m + 3))
    h.close()
