"""Ranking a long row through its compacted candidates.

With at most 64 ranked entries a row of more than 1024 keys is searched over the
keys at or above the smallest lane maximum; with more the whole row is searched.
Both rank the same rows here and must agree exactly: random scores, ties across
the cut, rows with too many or too few candidates for the list, probabilities
that underflow, and non-finite scores (equal bits in, equal order out)."""
import pytest
import torch

from oracle import routing as R
from route_check import check_rows

pytestmark = pytest.mark.gpu


def _rows(kind, Q, N, g):
    s = torch.randn(1, Q, N, generator=g)
    if kind == "ties":
        s = (s * 3).round() / 2
    elif kind == "equal":
        s = torch.zeros(1, Q, N)
    elif kind == "sorted":
        s = s.sort(-1, descending=True).values
    elif kind == "lane":  # one lane of the wave holds only keys of probability 0
        s[..., 5::64] = -200.0
    elif kind == "steep":
        s = s * 60
    elif kind == "plateau":  # 512 and 513 candidates: the list's last entry and one more
        s = s * 0.01 - 4
        for r in range(Q):
            s[0, r, torch.randperm(N // 64, generator=g)[:8, None] * 64 + torch.arange(64)] = 1.0
            if r % 2:
                s[0, r, (s[0, r] < 0).nonzero()[0]] = 1.0
    elif kind == "nonfinite":
        s[0, 0, 7], s[0, 1, 9], s[0, 2] = float("inf"), float("nan"), float("-inf")
    return s


@pytest.mark.parametrize("kind", ["random", "ties", "equal", "sorted", "lane", "steep", "plateau", "nonfinite"])
@pytest.mark.parametrize("N", [1025, 2048, 3000, 4096])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_candidates_rank_as_the_row(fsi, dev, kind, N, dtype):
    print(f"[case] route candidates {kind} {N} {dtype}", flush=True)
    s = _rows(kind, 7, N, torch.Generator().manual_seed(N)).to(dtype).to(dev)
    for causal, local, k_max in ((False, 0, 64), (False, 0, 5), (False, 3, 64), (True, 0, 64)):
        x = s if not causal else s.expand(1, 7, N)
        kw = dict(causal=causal, local_window_blocks=local, top_p=0.9, min_remote_blocks=2, max_remote_blocks=k_max)
        a = fsi.select_blocks(x, remote_capacity=k_max, **kw)
        b = fsi.select_blocks(x, remote_capacity=128, **kw)
        assert torch.equal(a.remote_counts, b.remote_counts)
        assert torch.equal(a.remote_indices, b.remote_indices[..., :k_max])


@pytest.mark.parametrize("N", [1030, 2000, 4096])
@pytest.mark.parametrize("keys", ["random", "repeated", "tiny", "wide"])
def test_scored_candidates_rank_as_the_row(fsi, dev, N, keys):
    """score_and_route: indices, counts and mass of the two searches agree exactly (fp64 sums of
    these masses are exact in either order), and with the oracle, whose normalisation and
    softmax are plain fp32 divisions, up to near-ties."""
    print(f"[case] scored candidates {keys} {N}", flush=True)
    g = torch.Generator().manual_seed(N + len(keys))
    q, k = torch.randn(2, 37, 16, generator=g), torch.randn(2, N, 16, generator=g)
    if keys == "repeated":
        k = k[:, torch.randint(0, 40, (N,), generator=g)].contiguous()
    elif keys == "tiny":  # norms on both sides of 2^-40, components under 2^-60, zero keys
        k = k * 2.0 ** torch.randint(-60, 0, (2, N, 1), generator=g)
        k[:, ::17] = 0
    elif keys == "wide":
        k = k * 2.0 ** torch.randint(-70, 30, (2, N, 16), generator=g)
    kw = dict(causal=False, local_window_blocks=0, top_p=0.9, min_remote_blocks=4, max_remote_blocks=64, return_mass=True)
    ia, ca, ma = fsi.score_and_route(q.to(dev), k.to(dev), remote_capacity=64, **kw)
    ib, cb, mb = fsi.score_and_route(q.to(dev), k.to(dev), remote_capacity=128, **kw)
    assert torch.equal(ca, cb) and torch.equal(ma, mb) and torch.equal(ia, ib[..., :64])
    ora = R.select_route(R.cosine_scores_f32(q, k), causal=False, top_p=0.9, min_remote_blocks=4, max_remote_blocks=64,
                         remote_capacity=64)
    bad = check_rows(ia, ca, ora, torch.ones(37, N, dtype=torch.bool), 1e-6, 1e-5)
    assert not bad, bad
    cnt = ora["remote_counts"].long()
    want = ora["cumulative"].gather(2, (cnt - 1)[..., None])[..., 0]  # at least 4 are taken
    same = ca.cpu().long() == cnt
    assert same.any() and torch.allclose(ma.cpu()[same], want[same], atol=2e-6)
