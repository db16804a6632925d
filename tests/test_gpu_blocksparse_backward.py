"""Gradients of the 2-D tile-sparse matmul (block_matmul.py:381-392) on the HIP backward
against fp64: every tile form it takes (64 and multiples of 128, each side), one and
several row groups, ragged rows, empty and dense masks; the tilings it does not take and
a differentiated backward run the library form and give the same."""
import pytest
import torch

from oracle import blocksparse as BS
from oracle import pattention as P

pytestmark = pytest.mark.gpu

CASES = [  # M, K, N, block_k, block_n, density, groups, rows_per_group
    (1, 128, 128, 128, 128, 1.0, 1, 1),         # smallest: one row, one tile
    (33, 64, 64, 64, 64, 1.0, 1, 33),           # one tile of 64: half an output tile
    (130, 192, 320, 64, 64, 0.4, 1, 130),       # N and K end inside an output tile, quarters
    (300, 256, 384, 128, 64, 0.5, 3, 128),      # quarters: 64-row groups of dW, 128-wide tiles
    (300, 320, 256, 64, 128, 0.5, 3, 128),      # two k blocks per column tile
    (257, 256, 256, 64, 64, 0.5, 2, 256),       # last group of one row
    (100, 256, 512, 128, 256, 0.5, 4, 128),     # groups past the rows
    (640, 512, 768, 256, 128, 0.3, 5, 128),
    (256, 256, 256, 128, 128, 0.0, 2, 128),     # nothing active
    (512, 3072, 3072, 128, 128, 0.25, 4, 128),  # 576 output tiles of dW: heaviest-first order
    (256, 3072, 3072, 64, 64, 0.2, 2, 128),     # and its quarters
    (96, 192, 96, 64, 48, 0.5, 1, 96),          # not taken: n blocks of 48
    (256, 256, 256, 32, 64, 0.5, 2, 128),       # not taken: k blocks of 32
    (257, 256, 256, 128, 64, 0.5, 5, 128),      # two groups past the rows
]


def _inputs(case, dtype, dev):
    M, K, N, bk, bn, density, groups, rpg = case
    g = torch.Generator().manual_seed(M + K + N + bk)
    x, w, dy = (torch.randn(*s, generator=g).to(dtype) for s in ((M, K), (N, K), (M, N)))
    mask = torch.rand(groups, (K // bk) * (N // bn), generator=g) < density
    return x, w, dy, mask


def _expected(case, x, w, dy, mask):
    M, K, N, bk, bn, _, groups, rpg = case
    dx, dw = torch.zeros(M, K, dtype=torch.float64), torch.zeros(N, K, dtype=torch.float64)
    for i in range(groups):
        r = slice(min(M, i * rpg), min(M, (i + 1) * rpg)) if groups > 1 else slice(0, M)
        em = BS.expand_tile_mask(mask[i], N, K, bk, bn).double()
        dx[r] = dy[r].double() @ (w.double() * em)
        dw += (dy[r].double().t() @ x[r].double()) * em
    return dx, dw


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[f"b{i}" for i in range(len(CASES))])
def test_blockwise_matmul_gradients(fsi, dev, case, dtype):
    print(f"[case] blockwise_matmul backward {case} {dtype}", flush=True)
    M, K, N, bk, bn, density, groups, rpg = case
    x, w, dy, mask = _inputs(case, dtype, dev)
    xd, wd = x.to(dev).requires_grad_(), w.to(dev).requires_grad_()
    y = fsi.blockwise_matmul(xd, wd, mask.to(dev), bk, bn, rows_per_group=rpg)
    got = torch.autograd.grad(y, (xd, wd), dy.to(dev))
    taken = bk % 64 == 0 and bn in (64, 128, 256)
    # fp32 sums rounded once to bf16 (2^-9 relative per value); the library form of
    # several groups also rounds each group's partial sum
    tol = 1e-5 if dtype == torch.float32 else 2e-3 if taken else 5e-3
    for a, e in zip(got, _expected(case, x, w, dy, mask)):
        assert a.dtype == dtype
        if e.any():
            assert P.rel_l2(a.cpu().float(), e.float()) <= tol
        else:
            assert not a.any()


def test_blockwise_matmul_gradient_forms(fsi, dev):
    """A strided and misaligned dy, one wanted gradient only, and a backward that is
    differentiated itself give what the plain backward gives."""
    case = (200, 256, 384, 64, 128, 0.5, 2, 128)
    M, K, N, bk, bn, _, _, rpg = case
    x, w, dy, mask = _inputs(case, torch.float32, dev)
    x, w, dy, mask = (t.to(dev) for t in (x, w, dy, mask))
    dx, dw = (t.to(dev, torch.float32) for t in _expected(case, x.cpu(), w.cpu(), dy.cpu(), mask.cpu()))

    def grads(want, grad, **kw):
        xd, wd = x.clone().requires_grad_("x" in want), w.clone().requires_grad_("w" in want)
        y = fsi.blockwise_matmul(xd, wd, mask, bk, bn, rows_per_group=rpg)
        return torch.autograd.grad(y, [t for t in (xd, wd) if t.requires_grad], grad, **kw)

    odd = torch.zeros(M * N + 1, device=dev)[1:].view(M, N).copy_(dy)  # 4-byte aligned
    wide = torch.zeros(M, 2 * N, device=dev)[:, ::2].copy_(dy)
    for form in (odd, wide, dy.t().contiguous().t()):
        a, b = grads("xw", form)
        assert P.rel_l2(a, dx) <= 1e-5 and P.rel_l2(b, dw) <= 1e-5
    assert P.rel_l2(grads("x", dy)[0], dx) <= 1e-5
    assert P.rel_l2(grads("w", dy)[0], dw) <= 1e-5
    a, b = grads("xw", dy.clone().requires_grad_(), create_graph=True)
    assert a.requires_grad and P.rel_l2(a.detach(), dx) <= 1e-5 and P.rel_l2(b.detach(), dw) <= 1e-5
