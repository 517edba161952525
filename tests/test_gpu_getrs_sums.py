"""PDGETRS with more than 16 right-hand sides: sums of at most 128 products, each taken
from B by itself.  The last row solved takes 2^53 * 1, which B holds too, from the
first of 256 solved values and 1 * 1 from each of the last 128.  Exactly -128 is left;
in one sum the ones would all be rounded away.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nrhs", [17, 40])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("upper", [False, True])
def test_sums_of_a_block(upper, trans, nrhs):
    from scalapack_amd.device import Handle
    n = 257
    e = np.eye(n)  # op(triangle), its rows in the order they are solved
    e[256, 0] = 2.0 ** 53
    e[256, 128:256] = 1.0
    b = np.ones(n)
    b[256] = 2.0 ** 53
    x = b.copy()
    x[256] = -128.0
    if upper == (trans == "N"):  # U and L^T: from the last row up
        e, b, x = e[::-1, ::-1], b[::-1], x[::-1]
    a = e if trans == "N" else e.T
    da = torch.from_numpy(np.ascontiguousarray(a.T)).cuda()
    db = torch.from_numpy(np.tile(b, (nrhs, 1))).cuda()
    dp = torch.arange(1, n + 1, dtype=torch.int32, device="cuda")
    h = Handle()
    print(f"[gpu] getrs sums upper={upper} {trans} nrhs={nrhs}", flush=True)
    h.dgetrs_trans(trans, n, nrhs, da, n, dp, db, n)
    h.close()
    assert np.array_equal(db.cpu().numpy(), np.tile(x, (nrhs, 1)))
