"""Rules that choose between kernels, and what they ask of a step's workspace (no GPU: the library's host code alone)."""
import pytest

from gibbs_amd.ops.lib import library


@pytest.mark.parametrize("n,o", [(333, 1024), (700, 512), (1194, 1024)])
def test_float32_products_ask_for_a_workspace_where_their_kernel_uses_it(n, o):
    """Few tiles of a long inner size share their stretches through one.  Rows that are no whole 16 bytes take the plain kernel, which has
    no use for it."""
    assert library().gibbs_gemm_f32_workspace(n, o, 2052) > 0
    assert [library().gibbs_gemm_f32_workspace(n, o, 2052 + k) for k in (1, 2, 3)] == [0, 0, 0]
