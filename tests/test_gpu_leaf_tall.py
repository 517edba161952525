"""Panel leaves of more workgroups than one die runs, up to the most that a leaf may
have, and the narrow ones that are cut like them: every pivot search ties (the
matrices of test_gpu_leaf), also between workgroups 64 and up.
"""
import pytest

from test_gpu_leaf import check, incidence

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m,w", [(1025, 8), (2049, 7), (1025, 16), (16385, 8), (33000, 3), (33000, 16),
                                 (65537, 8), (65537, 16), (131072, 1), (131072, 12), (131073, 5),
                                 (131073, 16), (33000, 17), (65536, 32), (66000, 17), (66000, 32),
                                 (131072, 32)])
def test_tall_leaf_exact(m, w):
    from scalapack_amd.device import Handle
    h = Handle(nb=64)
    check(h, incidence(m, w, seed=100 * w + m))
    h.close()
