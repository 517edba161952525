"""gemm_tile_sub's launches that no size of the public entry points reaches quickly:
grids smaller than the number of tiles (only the trailing update's kernel takes
several tiles a workgroup; any other has to get a workgroup each), and leading
dimensions whose offsets need 64 bits.  Whole numbers: results are exact.
"""
import ctypes
import shutil
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def gemm():
    from scalapack_amd import _lib
    if not shutil.which("nm"):
        pytest.skip("nm not found")
    names = subprocess.run(["nm", "-D", "--defined-only", str(_lib.PKG / "libscalapack_amd.so")],
                           check=True, capture_output=True, text=True).stdout.split()
    fn = getattr(_lib.load(), next(n for n in names if "gemm_tile_subIdE" in n))
    p, i, b = ctypes.c_void_p, ctypes.c_int, ctypes.c_bool
    fn.restype = None
    fn.argtypes = [b, i, i, i, p, i, p, i, p, i, p, b, i, b, p, b]

    def call(m, n, k, a, lda, b, ldb, c, ldc, ta=False, trailing=False, max_wgs=0, solve=False):
        print(f"[gpu] gemm launch {m} {n} {k} ta={ta} trailing={trailing} wgs={max_wgs}", flush=True)
        fn(ta, m, n, k, a.data_ptr(), lda, b.data_ptr(), ldb, c.data_ptr(), ldc, None, trailing,
           max_wgs, False, None, solve)
        torch.cuda.synchronize()
    return call


def whole(r, c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-9, 10, (c, r), device="cuda", generator=g).double()


def product(a, b):
    """A B of column-major whole-number matrices, computed on the host."""
    return torch.from_numpy(b.cpu().numpy() @ a.cpu().numpy()).cuda()


@pytest.mark.parametrize("trailing,solve", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n,k,wgs", [(640, 640, 48, 8), (1000, 700, 16, 24), (900, 20, 33, 9),
                                       (640, 640, 16, 7), (640, 640, 16, 1000)])
def test_small_grids(gemm, m, n, k, wgs, trailing, solve):
    a, b, c = whole(m, k, 1), whole(k, n, 2), whole(m, n, 3)
    want = c - product(a, b)
    gemm(m, n, k, a, m, b, k, c, m, trailing=trailing, max_wgs=wgs, solve=solve)
    assert torch.equal(c, want)


@pytest.mark.parametrize("ta,trailing,solve", [(False, False, False), (False, True, False),
                                               (False, False, True), (True, False, True)])
@pytest.mark.parametrize("n", [20, 65])
def test_offsets_beyond_32_bits(gemm, n, ta, trailing, solve):
    m, k, ld = 130, 35, 7_000_000  # 80 columns of 56 MB
    assert 80 * ld * 8 > 2 ** 32
    a, b, c = whole(m, k, 1), whole(k, n, 2), whole(m, n, 3)
    want = c - product(a, b)
    src = a.t().contiguous() if ta else a
    wide = torch.full((src.shape[0], ld), np.nan, dtype=torch.float64, device="cuda")
    wide[:, :src.shape[1]] = src
    widb = torch.full((n, ld), np.nan, dtype=torch.float64, device="cuda")
    widb[:, :k] = b
    torch.cuda.synchronize()
    gemm(m, n, k, wide, ld, widb, ld, c, m, ta=ta, trailing=trailing, solve=solve)
    assert torch.equal(c, want)
