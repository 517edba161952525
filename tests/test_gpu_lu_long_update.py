"""Trailing updates that outlast their panel (128 x 256 tiles, 64 x 64 at their borders)
and leaves beside long updates, of more than 64 workgroups: factors and IPIV equal bit
for bit to those of one stream, where every update takes 64 x 64 tiles and every leaf
stands alone; also with a persistent grid on part of the CUs.
"""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def factor(a0, m, n, lda, **params):
    from scalapack_amd.device import Handle
    a, p = a0.clone(), torch.zeros(min(m, n), dtype=torch.int32, device="cuda")
    h = Handle(**params)
    print(f"[gpu] dgetrf {m} x {n} {params}", flush=True)
    assert h.dgetrf(m, n, a, lda, p) == 0
    h.close()
    return a, p


# wide matrices: an update outlasts its panel from a moderate number of rows on
@pytest.mark.parametrize("m,n,lda,nb", [(8192, 50000, 8192, 64), (8260, 50100, 8264, 96),
                                        (8201, 50000, 8201, 64), (20480, 12000, 20480, 64),
                                        (20480, 24000, 20480, 64)])
def test_factors_equal_those_of_one_stream(m, n, lda, nb):
    g = torch.Generator(device="cuda").manual_seed(m)
    a0 = torch.randn(n, lda, dtype=torch.float64, device="cuda", generator=g)
    # a quarter of the entries in whole numbers: many ties, exact at first
    a0[:, ::4] = a0[:, ::4].round()
    want = factor(a0, m, n, lda, nb=nb, lookahead=0)
    for params in ({}, {"update_cus": 8}):
        got = factor(a0, m, n, lda, nb=nb, **params)
        assert torch.equal(got[1], want[1]) and torch.equal(got[0], want[0]), params
