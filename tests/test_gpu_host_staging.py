"""Host arrays on their way to the device and back in pieces of columns: one piece,
several, the last one ragged, a leading dimension beyond the rows, and a submatrix
whose surroundings stay as they are.

PDGETRF's factors from host arrays equal those of the device entry bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m,n,lld,off", [(1, 1, 1, 0), (5, 3, 9, 0), (100, 100, 100, 0),
                                         (130, 70, 300, 64), (724, 724, 724, 0), (725, 725, 730, 0),
                                         (3000, 400, 3001, 0), (20000, 53, 20000, 0)])
def test_pieces(m, n, lld, off):
    from scalapack_amd import api
    from scalapack_amd.device import Handle
    rng = np.random.default_rng(m + n)
    nb = 64
    big = np.asfortranarray(rng.standard_normal((lld + off, n + off)))
    want = big.copy()
    ctx = api.blacs_gridinit(1, 1)
    desc, _ = api.descinit(m + off, n + off, nb, nb, 0, 0, ctx, lld + off)
    k = min(m, n)
    ipiv = np.zeros(m + off + nb, np.int32)
    print(f"[gpu] pdgetrf host m={m} n={n} lld={lld + off} off={off}", flush=True)
    info = api.pdgetrf(m, n, big, off + 1, off + 1, desc, ipiv)
    assert info == 0

    h = Handle()
    sub = want[off:off + m, off:off + n]
    da = torch.from_numpy(np.ascontiguousarray(sub.T)).cuda()
    dp = torch.zeros(k, dtype=torch.int32, device="cuda")
    assert h.dgetrf(m, n, da, m, dp) == 0
    h.close()
    want[off:off + m, off:off + n] = da.cpu().numpy().T
    np.testing.assert_array_equal(big, want)
    np.testing.assert_array_equal(ipiv[off:off + k], dp.cpu().numpy() + off)
