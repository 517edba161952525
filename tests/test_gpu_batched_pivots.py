"""Pivot choice of the batched factorization where many rows share the largest
magnitude: A is a block diagonal of 8 x 8 Hadamard matrices (random signs) with its
rows shuffled over the whole matrix.  Every minor of such a block is a power of two
or zero times a common power of two, so elimination with partial pivoting is exact
in FP32 and FP64, and the factors and IPIV equal numpy's elimination bit for bit.
The sizes are the edges of a wave, of a panel and of one against two rows a thread.
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


def _shuffled_hadamard(n, rng):
    h2 = np.array([[1.0, 1.0], [1.0, -1.0]])
    h8 = np.kron(np.kron(h2, h2), h2)
    a = np.eye(n)
    for k in range(0, n - 7, 8):
        sr, sc = rng.choice([-1.0, 1.0], 8), rng.choice([-1.0, 1.0], 8)
        a[k:k + 8, k:k + 8] = sr[:, None] * h8[rng.permutation(8)] * sc
    return a[rng.permutation(n)]


def _eliminate(a):
    a = a.copy()
    n = a.shape[0]
    piv = np.zeros(n, np.int32)
    for j in range(n):
        p = j + int(np.argmax(np.abs(a[j:, j])))  # the first largest
        piv[j] = p + 1
        a[[j, p]] = a[[p, j]]
        a[j + 1:, j] /= a[j, j]
        hit = np.nonzero(a[j + 1:, j])[0] + j + 1
        a[hit, j + 1:] -= np.outer(a[hit, j], a[j, j + 1:])
    return a, piv


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("w", [8, 16, 32])
def test_ties(dev, w, prec):
    rng = np.random.default_rng(w)
    ns = [1, 8, 15, 16, 17, 33, 63, 64, 65, 130, 511, 512, 513, 529, 777, 1024]
    dt = np.float64 if prec == "fp64" else np.float32
    mats = [_shuffled_hadamard(n, rng) for n in ns]
    bufs = []
    for a in mats:
        buf = np.full((a.shape[0], a.shape[0] + 2), np.nan, dt)  # column major, lda = n + 2
        buf[:, :a.shape[0]] = a.T
        bufs.append(torch.from_numpy(buf).cuda())
    bs = [torch.ones(1, n, dtype=bufs[0].dtype, device="cuda") for n in ns]
    ps = [torch.zeros(n, dtype=torch.int32, device="cuda") for n in ns]
    ptr = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64).cuda()  # noqa: E731
    info = torch.full((len(ns),), -7, dtype=torch.int32, device="cuda")
    print(f"[gpu] batched ties w={w} {prec}", flush=True)
    w0 = dev.get("batched_w")
    dev.set("batched_w", w)
    try:
        dev.gesv_batched(prec, ns, [1] * len(ns), ptr(bufs), [n + 2 for n in ns], ptr(ps),
                         ptr(bs), ns, info)
    finally:
        dev.set("batched_w", w0)
    assert (info.cpu().numpy() == 0).all()
    for n, a, buf, p in zip(ns, mats, bufs, ps):
        lu, piv = _eliminate(a)
        got = buf.cpu().numpy()
        assert np.isnan(got[:, n:]).all()
        np.testing.assert_array_equal(p.cpu().numpy(), piv, err_msg=str(n))
        np.testing.assert_array_equal(got[:, :n].T, lu.astype(dt), err_msg=str(n))
