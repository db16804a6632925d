"""Backward of the block-sparse attention in bf16 (fsi_sparse_attn_bwd) at the edges of its
64 x 64 tiles against fp64: one head, pairs and odd groups of query heads per KV head, the
three ways a tile's weights are found (pattern blocks of a multiple of 64, of 16, other),
ragged and one-row sequences, more than 64 tiles, and rows that are only 4-element aligned."""
import math

import pytest
import torch

from oracle import attention as A
from oracle import pattention as P

pytestmark = pytest.mark.gpu

CASES = [  # B, Hq, Hkv, hd, T, block, window, cap, mode
    (1, 1, 1, 128, 1, 64, 64, 1, 0),      # one query, one key
    (1, 2, 1, 128, 65, 64, 7, 1, 0),      # a tile and one row
    (2, 6, 2, 128, 191, 64, 64, 2, 0),    # three heads a group: one head a workgroup
    (1, 8, 2, 64, 256, 128, 100, 2, 0),   # blocks of two tiles
    (1, 4, 1, 128, 130, 16, 20, 3, 0),    # classes per 16 x 16 sub-tile
    (1, 2, 2, 64, 150, 48, 33, 2, 0),     # sub-tiles, blocks across tiles
    (1, 2, 1, 32, 200, 24, 10, 3, 0),     # classes per element
    (1, 2, 1, 128, 100, 10, 5, 3, 0),
    (2, 2, 1, 128, 192, 64, 0, 3, 1),     # block lists, a block listed twice
    (1, 4, 2, 64, 160, 16, 0, 4, 1),
    (1, 2, 2, 32, 96, 8, 0, 4, 1),
    (1, 2, 1, 32, 4200, 64, 100, 2, 0),   # 66 tiles: a second list register
    (1, 3, 1, 64, 70, 64, 5, 1, 0),       # one head a workgroup, its waves sharing a tile's keys:
    (1, 1, 1, 128, 33, 16, 40, 3, 0),     # one key past a half
    (1, 1, 1, 64, 96, 32, 0, 1, 1),       # halves that no query attends
    (2, 3, 3, 32, 100, 10, 3, 2, 0),
    (1, 3, 1, 128, 200, 24, 0, 3, 1),
]


def _inputs(case, seed):
    B, Hq, Hkv, hd, T, blk, W, cap, mode = case
    g = torch.Generator().manual_seed(seed)
    q, k, v, dout = (torch.randn(B, h, T, hd, generator=g).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    nb = -(-T // blk)
    idx = torch.randint(0, nb, (B, nb, cap), generator=g, dtype=torch.int32)
    cnt = torch.randint(0, cap + 1, (B, nb), generator=g, dtype=torch.int32)
    if cap > 1:
        idx[0, nb - 1, :2] = 0
        cnt[0, nb - 1] = max(int(cnt[0, nb - 1]), 2)
    if mode == 1:
        cnt[0, 0] = 0  # rows that attend nothing
    return q, k, v, dout, idx, cnt


def _expected(case, q, k, v, dout, idx, cnt):
    B, Hq, Hkv, hd, T, blk, W, cap, mode = case
    w = A.sparse_mask(B, T, W, blk, idx, cnt) if mode == 0 else A.block_list_weights(B, T, blk, idx, cnt)
    leaf = [t.double().requires_grad_() for t in (q, k, v)]
    A.weighted_attention_f64(*leaf, w, 1.0 / math.sqrt(hd)).backward(dout.double())
    return [t.grad for t in leaf]


def _check(got, want):
    # D = dout . out takes the forward's bf16 output (2^-9 relative) and the gradients round
    # once more; P and dS are held to 2^-17
    for a, e in zip(got, want):
        if e.any():
            assert P.rel_l2(a.cpu().float(), e.float()) <= 1e-2
        else:
            # dP - D cancels: two fp32 sums of head_dim products of N(0, 1) values differ by at
            # most hd 2^-24 sum |dout v| < 128 * 6e-8 * 128, times |k| / sqrt(hd) < 0.5
            assert a.abs().max() <= 5e-4


@pytest.mark.parametrize("case", CASES, ids=[f"t{i}" for i in range(len(CASES))])
def test_sparse_attention_backward_bf16(fsi, dev, case):
    print(f"[case] sparse_attention backward {case}", flush=True)
    hd, blk, W, mode = case[3], case[5], case[6], case[8]
    q, k, v, dout, idx, cnt = _inputs(case, sum(case))
    leaf = [t.to(dev).requires_grad_() for t in (q, k, v)]
    out = fsi.sparse_attention(*leaf, idx.to(dev), cnt.to(dev), block=blk, mode=mode, window=W)
    got = torch.autograd.grad(out, leaf, dout.to(dev))
    _check(got, _expected(case, q, k, v, dout, idx, cnt))


@pytest.mark.parametrize("pad", [4, 1])
def test_sparse_attention_backward_short_alignment(fsi, dev, pad):
    """Operands whose rows start at a multiple of 4 elements (8 bytes) or of one element
    only (copied into aligned ones) give the same gradients."""
    case = (1, 2, 1, 64, 130, 64, 40, 2, 0)
    hd, blk, W = case[3], case[5], case[6]
    q, k, v, dout, idx, cnt = _inputs(case, 5)

    def odd(t):
        wide = torch.zeros(*t.shape[:-1], hd + pad, dtype=t.dtype, device=dev)
        wide[..., pad:] = t.to(dev)
        return wide[..., pad:]

    out = fsi.sparse_attention(q.to(dev), k.to(dev), v.to(dev), idx.to(dev), cnt.to(dev), block=blk, window=W)
    got = fsi.attention._sparse_attention_bwd(odd(q), odd(k), odd(v), out, dout.to(dev), idx.to(dev), cnt.to(dev), 2,
                                              blk, 0, W, 1.0 / math.sqrt(hd))
    _check(got, _expected(case, q, k, v, dout, idx, cnt))
