"""The operands that the sparse attention's bf16 backward kernels are handed (CPU only)."""
import pytest
import torch

T_STRIDE = 4 * 64
CASES = {  # shape, strides, first element, copied
    "packed": ((2, 4, 5, 64), (1280, 320, 64, 1), 0, False),
    "heads inside": ((2, 4, 5, 64), (5 * T_STRIDE, 64, T_STRIDE, 1), 0, False),
    "start of 4": ((2, 4, 5, 64), (1280, 320, 64, 1), 4, True),
    "rows of 68": ((1, 2, 5, 64), (680, 340, 68, 1), 0, True),
    "one row": ((1, 1, 1, 64), (68, 68, 68, 1), 0, True),
    "other head_dim": ((1, 2, 5, 40), (430, 215, 43, 1), 3, False),
}


@pytest.mark.parametrize("kind", CASES)
def test_rows_are_aligned(fsi, kind):
    shape, strides, start, copied = CASES[kind]
    t = torch.arange(4096).bfloat16().as_strided(shape, strides, start)
    y = fsi.attention._bwd_operand(t)
    assert torch.equal(y, t) and (y is not t) == copied
    if shape[3] == 64:
        assert y.data_ptr() % 16 == 0 and not any(s % 8 for s in y.stride()[:3])
    assert fsi.attention._bwd_operand(t.float()).shape == shape
