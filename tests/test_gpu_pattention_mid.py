"""Pattention of 65 .. 255 tokens (csrc/pattention_mid.hip) against the oracle: both ends of the
range and of its token tiles, the three rounding points, whole and listed blocks, both tile
counts and several splits, an out-of-range block id, and shapes that keep to the other kernels."""
import pytest
import torch

from oracle import pattention as P

pytestmark = pytest.mark.gpu

TOL = 2e-3  # rel-L2, the bar of the other bf16 Pattention kernels

CASES = [  # M, K, D_out, block_n, n_blocks, active (None: all), rounding
    (65, 4096, 256, 64, 80, 64, "fused"),
    (128, 4096, 512, 64, 64, None, "eager"),
    (129, 2048, 2048, 64, 112, 100, "fp32"),   # 100 steps of the down projection: two splits at least
    (255, 4096, 1024, 128, 40, 32, "fused"),
    (100, 3200, 256, 64, 80, 64, "fused"),     # 50 steps: two splits, uneven rings
    (144, 4096, 1040, 64, 64, None, "fused"),  # output columns of an odd number of tiles: other kernels
    (100, 4104, 256, 64, 64, None, "fused"),   # K no multiple of 64: other kernels
    (200, 4096, 512, 32, 128, None, "fused"),  # blocks of 32: other kernels
    (100, 2048, 2048, 64, 96, 24, "fused"),    # small weights: other kernels
]


def _inputs(case):
    M, K, D, bn, nb, n_act, _ = case
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g).bfloat16()
    kg, ku = (torch.randn(nb * bn, K, generator=g).mul_(K ** -0.5).bfloat16() for _ in range(2))
    vt = torch.randn(D, nb * bn, generator=g).mul_(0.05).bfloat16()
    act = None if n_act is None else torch.randperm(nb, generator=g)[:n_act].to(torch.int32)
    return x, kg, ku, vt, act


def _expected(case, x, kg, ku, vt, act):
    M, K, D, bn, nb, _, rounding = case
    blocks = torch.arange(nb) if act is None else act
    if rounding == "fp32":
        return P.pattention_fp32_act(x, kg, vt.t().contiguous(), ku, blocks, "swiglu", bn)
    return P.mlp_eval_forward(x, kg, ku, vt.t().contiguous(), blocks, bn, fused=(rounding == "fused"))


@pytest.mark.parametrize("case", CASES, ids=[f"m{i}" for i in range(len(CASES))])
def test_mid_pattention(fsi, dev, case):
    print(f"[case] pattention mid {case}", flush=True)
    x, kg, ku, vt, act = _inputs(case)
    got = fsi.pattention_forward(x.to(dev), kg.to(dev), ku.to(dev), vt.to(dev).t(),
                                 None if act is None else act.to(dev), case[3], "swiglu", case[6])
    assert P.rel_l2(got.cpu().float(), _expected(case, x, kg, ku, vt, act).float()) <= TOL


def test_mid_pattention_block_out_of_range(fsi, dev):
    """An id past the blocks contributes nothing and is recorded."""
    case = (80, 4096, 512, 64, 80, 66, "fused")
    x, kg, ku, vt, act = _inputs(case)
    bad = act.clone()
    bad[3], bad[7] = 80, -1
    err = fsi._lib.error_word(dev)
    err.zero_()
    got = fsi.pattention_forward(x.to(dev), kg.to(dev), ku.to(dev), vt.to(dev).t(), bad.to(dev), 64, "swiglu", "fused")
    assert int(err[0].item()) == fsi._lib.FSI_ERR_INDEX_RANGE
    err.zero_()
    keep = act[[i for i in range(66) if i not in (3, 7)]]
    assert P.rel_l2(got.cpu().float(), _expected(case, x, kg, ku, vt, keep).float()) <= TOL


def test_mid_pattention_strided_rows(fsi, dev):
    """Token rows of a wider tensor and an output slice."""
    case = (150, 4096, 1024, 64, 80, 64, "fused")
    x, kg, ku, vt, act = _inputs(case)
    wide = torch.zeros(150, 4096 + 8, dtype=torch.bfloat16, device=dev)
    wide[:, 8:] = x.to(dev)
    out = torch.zeros(150, 1024 + 3, dtype=torch.bfloat16, device=dev)
    fsi.pattention_forward(wide[:, 8:], kg.to(dev), ku.to(dev), vt.to(dev).t(), act.to(dev), 64, "swiglu", "fused",
                           out=out[:, 3:])
    assert P.rel_l2(out[:, 3:].cpu().float(), _expected(case, x, kg, ku, vt, act).float()) <= TOL
    assert not out[:, :3].any()
