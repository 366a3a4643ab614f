"""What the dense product's plan chooses, host arithmetic."""

import pytest

from neuropress_amd import _lib


@pytest.mark.parametrize("m,n,k,parts", [(548, 320, 9728, 7), (444, 352, 9856, 8), (601, 432, 9344, 6), (512, 512, 8192, 6)])
def test_long_k_over_few_tiles(m, n, k, parts):
    """As many parts of K as make one round of 64 x 128 tiles, up to eight: the tile in two groups.  With wide tiles alone 5, 6, 3 and 4 parts, 8 to 15 % slower."""
    assert _lib.load().npamd_dense_gemm_workspace_bytes(m, n, k) == parts * m * n * 4
