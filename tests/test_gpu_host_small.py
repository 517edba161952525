"""Host arrays at the edges of the small ones, which are packed in ordinary memory: one
column, two, and the first that takes more than 1 MB at the device's leading dimension.
"""
import pytest

import test_gpu_host_staging as staging

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,lld,off", [(1, 2, 4, 64), (2, 1, 2, 0), (70, 1, 71, 64), (300000, 1, 300000, 0),
                                         (70, 2, 70, 64), (361, 341, 361, 0), (361, 342, 365, 64)])
def test_small_pieces(m, n, lld, off):
    staging.test_pieces(m, n, lld, off)
