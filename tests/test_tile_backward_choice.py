"""Which tile-sparse matmul backward calls go to the HIP kernels (CPU only)."""
import pytest
import torch


@pytest.mark.parametrize("N,K,taken", [(64, 64, True), (64, 64 * 65535, True), (64, 64 * 65536, False),
                                       (2048 * 128, 128, True), (128 * 65536, 128, False)])
def test_wide_weights_keep_the_library(fsi, N, K, taken):
    """fsi_blockwise_matmul_bwd lays its transposes out over at most 65535 columns of 64."""
    block_n = 64 if N == 64 else 128 if N == 2048 * 128 else 128 * 64
    assert fsi.block_matmul._tile_bwd_supported(100, N, K, 1, 100, 64 if K % 128 else 128, block_n) == taken


@pytest.mark.parametrize("M,groups", [(100, 1), (128, 1), (129, 3)])
def test_groups_past_the_rows_are_not_padded_for(fsi, M, groups, monkeypatch):
    """A group much larger than the rows would have its scratch padded to its size."""
    seen = []

    def op(x2d, weight, dy, m8, block_k, block_n, rpg, want_dx, want_dw):
        seen.append(m8.shape[0])
        return torch.zeros_like(x2d), torch.zeros_like(weight)

    monkeypatch.setattr(fsi.block_matmul, "_blockwise_bwd_op", op)
    monkeypatch.setattr(fsi.block_matmul, "_blockwise_op", lambda x, w, *a: x @ w.t())
    x, w = torch.ones(M, 64, requires_grad=True), torch.ones(64, 64, requires_grad=True)
    fsi.block_matmul._BlockwiseMatmulFn.apply(x, w, torch.ones(3, 1, dtype=torch.uint8), 64, 64, 128).sum().backward()
    assert seen == [groups]
