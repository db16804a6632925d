"""Which tile-sparse matmul backward calls go to the HIP kernels (CPU only)."""
import pytest


@pytest.mark.parametrize("N,K,taken", [(64, 64, True), (64, 64 * 65535, True), (64, 64 * 65536, False),
                                       (2048 * 128, 128, True), (128 * 65536, 128, False)])
def test_wide_weights_keep_the_library(fsi, N, K, taken):
    """fsi_blockwise_matmul_bwd lays its transposes out over at most 65535 columns of 64."""
    block_n = 64 if N == 64 else 128 if N == 2048 * 128 else 128 * 64
    assert fsi.block_matmul._tile_bwd_supported(100, N, K, 1, 100, 64 if K % 128 else 128, block_n) == taken
