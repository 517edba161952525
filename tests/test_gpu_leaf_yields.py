"""Panel leaves that take more than a quarter of a die and so give way when their
workgroups do not all get to run: made to do so at their first look (patience 0), and
two handles at a time from two threads.  Exact matrices as in test_gpu_leaf.
"""
import threading

import numpy as np
import pytest

from test_gpu_leaf import check, incidence

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m", [8200, 16500, 32768])
@pytest.mark.parametrize("w", [2, 9, 17, 32])
def test_gives_way_at_once(m, w):
    from scalapack_amd.device import Handle
    h = Handle(nb=64, panel_patience=0)
    for seed in range(3):  # the mailbox changes regions from leaf to leaf
        check(h, incidence(m, w, seed=100 * w + m + seed))
    h.set("panel_patience", 200)
    check(h, incidence(m, w, seed=w + m))
    h.close()


def test_two_handles_at_once():
    from scalapack_amd.device import Handle
    m, n, passes = 20000, 64, 20
    a0 = [torch.randn(n, m, dtype=torch.float64, device="cuda",
                      generator=torch.Generator(device="cuda").manual_seed(s)) for s in (1, 2)]
    want = []
    h = Handle(nb=64)
    for a in a0:
        f, p = a.clone(), torch.zeros(n, dtype=torch.int32, device="cuda")
        assert h.dgetrf(m, n, f, m, p) == 0
        want.append((f, p))
    h.close()
    copies = [[a.clone() for _ in range(passes)] for a in a0]
    pivots = [[torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(passes)] for _ in a0]
    infos = [[], []]
    torch.cuda.synchronize()
    print("[gpu] two handles at once", flush=True)

    def work(i):
        hi = Handle(stream=None, nb=64)
        for a, p in zip(copies[i], pivots[i]):
            infos[i].append(hi.dgetrf(m, n, a, m, p))
        hi.close()

    threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in (0, 1):
        assert infos[i] == [0] * passes
        for a, p in zip(copies[i], pivots[i]):
            assert np.array_equal(a.cpu().numpy(), want[i][0].cpu().numpy())
            assert np.array_equal(p.cpu().numpy(), want[i][1].cpu().numpy())
