"""Rules that choose between kernels, and what they ask of a step's workspace (no GPU: the library's host code alone)."""
import pytest

from gibbs_amd.ops.lib import library


@pytest.mark.parametrize("n,o", [(333, 1024), (700, 512), (1194, 1024)])
def test_float32_products_ask_for_a_workspace_where_their_kernel_uses_it(n, o):
    """Few tiles of a long inner size share their stretches through one.  Rows that are no whole 16 bytes take the plain kernel, which has
    no use for it."""
    assert library().gibbs_gemm_f32_workspace(n, o, 2052) > 0
    assert [library().gibbs_gemm_f32_workspace(n, o, 2052 + k) for k in (1, 2, 3)] == [0, 0, 0]


# us, measured without and with the stretches shared
@pytest.mark.parametrize("n,o,i,alone,shared", [
    (333, 1024, 4608, 71.3, 40.8), (1194, 1024, 2048, 56.4, 50.0), (333, 4096, 2048, 61.1, 58.9), (400, 4096, 2048, 61.5, 67.4),
    (1500, 1024, 2048, 58.0, 55.9), (1700, 1024, 2048, 59.0, 64.6), (1600, 1024, 2560, 69.2, 72.9), (1600, 1024, 3072, 82.2, 84.1),
    (1600, 1024, 4608, 119.1, 116.5), (800, 2048, 2048, 59.0, 63.2), (150, 3072, 2048, 36.1, 35.0), (65, 2048, 8192, 62.1, 61.1),
    (2048, 256, 4096, 64.9, 39.0)])
def test_float32_products_share_their_stretches_where_that_is_faster(n, o, i, alone, shared):
    assert (library().gibbs_gemm_f32_workspace(n, o, i) > 0) == (shared < alone)
