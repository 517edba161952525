"""PDGETRS with many right-hand sides on a device with no memory for its whole
workspace: fewer columns at a time, the same bits, and the handle goes on working.
"""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_fewer_columns_at_a_time():
    from scalapack_amd.device import Handle
    n, nrhs, leave = 8192, 1024, 40 << 20  # the workspace is 64 MB
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g) / n
    a.diagonal().add_(1)
    p = torch.arange(1, n + 1, dtype=torch.int32, device="cuda")
    b0 = torch.randn(nrhs, n, dtype=torch.float64, device="cuda", generator=g)
    want, b = b0.clone(), b0.clone()
    h = Handle()
    h.dgetrs(n, nrhs, a, n, p, want, n)
    h.close()
    h = Handle()
    h.dgetrs(n, 1, a, n, p, b, n)  # what the handle needs for itself
    b.copy_(b0)
    torch.cuda.synchronize()
    held = []
    try:
        while True:
            size = min(torch.cuda.mem_get_info()[0] - leave, 64 << 30)
            if size < 1 << 20:
                break
            held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
    except torch.cuda.OutOfMemoryError:
        pass
    free = torch.cuda.mem_get_info()[0]
    print(f"[gpu] getrs with {free >> 20} MB free", flush=True)
    try:
        if not 36 << 20 <= free <= 60 << 20:
            pytest.skip("could not leave the memory that the test is about")
        h.dgetrs(n, nrhs, a, n, p, b, n)
    finally:
        del held
        torch.cuda.empty_cache()
    assert torch.equal(b, want)
    b.copy_(b0)
    h.dgetrs(n, nrhs, a, n, p, b, n)
    h.close()
    assert torch.equal(b, want)
