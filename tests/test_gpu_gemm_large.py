"""C -= A B of shapes that take 128 x 128 or 128 x 256 tiles (FP64) and 128 x 128 tiles
(FP32), with and without borders, and unaligned ones that do not.  Whole-number
operands: every sum is exact (FP32: below 2^24), and nothing outside C may change.
"""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def whole(rows, cols, lo, hi, ld, fill, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.full((cols, ld), fill, dtype=dt, device="cuda")
    t[:, :rows] = torch.randint(lo, hi + 1, (cols, rows), device="cuda", generator=g).to(dt)
    return t


# 2048: 256 tiles of 128 x 128; 4096: 512 of 128 x 256; 1536: 144 of 128 x 128 in FP32
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("m,n,k,pad", [(2048, 2048, 512, 0), (2048, 2048, 528, 4), (2050, 2177, 512, 2),
                                       (2048, 2048, 512, 1), (2048, 2048, 520, 0), (4096, 4096, 1024, 0),
                                       (4100, 4300, 1024, 4), (4096, 4096, 1024, 3), (1536, 1536, 928, 0),
                                       (1600, 1537, 1024, 0), (4096, 4096, 512, 0)])
def test_exact(prec, m, n, k, pad):
    from scalapack_amd.device import Handle
    dt = torch.float64 if prec == "fp64" else torch.float32
    nan = float("nan")
    a = whole(m, k, -9, 9, m + pad, nan, dt, 1)
    b = whole(k, n, -9, 9, k + pad, nan, dt, 2)
    c = whole(m, n, -9, 9, m + pad, 5.0, dt, 3)
    want = c.double()
    want[:, :m] -= b[:, :k].double() @ a[:, :m].double()
    h = Handle()
    print(f"[gpu] gemm {prec} {m} {n} {k} pad {pad}", flush=True)
    if prec == "fp64":
        h.dgemm_sub(m, n, k, a, m + pad, b, k + pad, c, m + pad)
    else:
        h.gemm_lowp_sub(m, n, k, a, m + pad, b, k + pad, c, m + pad, prec="fp32")
    h.close()
    assert torch.equal(c.double(), want)
