"""fp32 decode attention on both sides of the split-length rule.

Up to 2560 waves of 96 keys a call takes 32 keys a wave, above it 96; the
sequences here end inside and at the edge of a 32-key, a 96-key and a 16-key
piece, one sees a single key.  Bound: a probability carries the fp32 rounding of
a head_dim-term product (|s| <= 8 here) and of exp2, about 1e-6 relative, and
the sums over at most 3000 keys average further roundings, so rel-L2 against
fp64 stays under 1e-5."""
import pytest
import torch

from oracle import attention as A
from oracle import pattention as Pt

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, hd, max_seq, window, page, pages a sequence
    (1, 1, 1, 64, 40, 64, 16, 0),
    (2, 8, 2, 128, 700, 95, 64, 3),
    (4, 12, 2, 64, 1024, 97, 32, 5),
    (3, 34, 2, 128, 600, 33, 50, 4),  # 17 heads a group: two head blocks
    (5, 8, 8, 128, 6400, 2600, 64, 6),  # 5 x 8 x 32 waves: short splits, the merge's waves share 94
    (20, 32, 32, 64, 400, 300, 16, 5),  # 20 x 32 x 4 = 2560 waves: the last short one
    (20, 32, 32, 64, 400, 300, 16, 6),  # 20 x 32 x 5 waves: the long splits
]


@pytest.mark.parametrize("case", CASES, ids=[f"c{i}" for i in range(len(CASES))])
def test_split_length(fsi, dev, case):
    B, Hq, Hkv, hd, S, W, page, n_pages = case
    print(f"[case] fp32 decode splits {case}", flush=True)
    g = torch.Generator().manual_seed(B * 100 + hd)
    k, v = (torch.randn(B, Hkv, S, hd, generator=g) for _ in range(2))
    q = torch.randn(B, Hq, hd, generator=g)
    c = fsi.FovealKVCache(B, S, Hkv, hd, 16, page, dev, torch.float32, paged=False)
    c.load_dense(k.to(dev), v.to(dev))
    pos = [S - 1, 0, W - 1, min(S - 1, W + 31), S // 2][:B] + [S - 2] * max(0, B - 5)
    pages = [list(range(n_pages - (b % 2 if n_pages else 0))) for b in range(B)]
    rp = torch.full((B, max(1, n_pages)), -1, dtype=torch.int32)
    for b, p in enumerate(pages):
        rp[b, :len(p)] = torch.tensor(p, dtype=torch.int32)
    cnt = torch.tensor([len(p) for p in pages], dtype=torch.int32)
    out = fsi.decode_attention(q.to(dev), c, pos=torch.tensor(pos).to(dev), window=W,
                               remote_pages=rp.to(dev), remote_counts=cnt.to(dev), scale=hd ** -0.5)
    ref = A.decode_attention_f64(q.double(), k, v, pos, W, pages, page, hd ** -0.5)
    assert Pt.rel_l2(out.cpu().float(), ref.float()) <= 1e-5
