"""IPIV of a batched system whose column has a NaN on the diagonal and zeros below it:
no pivot, so INFO is that column, no rows are interchanged and IPIV says so.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("w", [8, 32])
def test_ipiv_names_the_interchanges_made(prec, w):
    from scalapack_amd.device import Handle
    dt = np.float64 if prec == "fp64" else np.float32
    where = [(3, 0), (3, 1), (70, 10), (70, 66), (600, 5), (600, 590)]
    mats = []
    for n, j in where:
        a = np.eye(n, dtype=dt)
        a[j, j] = np.nan
        a[:j, j + 1:] = 0.5
        mats.append(a)
    fa = [torch.from_numpy(np.ascontiguousarray(a.T)).cuda() for a in mats]
    fb = [torch.ones(1, len(a), dtype=fa[0].dtype, device="cuda") for a in mats]
    ps = [torch.zeros(len(a), dtype=torch.int32, device="cuda") for a in mats]
    ptr = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64).cuda()  # noqa: E731
    info = torch.full((len(mats),), -7, dtype=torch.int32, device="cuda")
    ns = [len(a) for a in mats]
    h = Handle(batched_w=w)
    print(f"[gpu] batched NaN pivot {prec} w={w}", flush=True)
    h.gesv_batched(prec, ns, [1] * len(ns), ptr(fa), ns, ptr(ps), ptr(fb), ns, info)
    h.close()
    assert info.cpu().tolist() == [j + 1 for _, j in where]
    for (n, j), a, f, p in zip(where, mats, fa, ps):
        assert np.array_equal(p.cpu().numpy(), np.arange(1, n + 1)), (n, j)
        assert np.array_equal(f.cpu().numpy().T, a, equal_nan=True), (n, j)
