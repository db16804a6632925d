"""Training forward / backward of FovealPattentionMLP on csrc/mlp_train.hip at the edges of
its kernels against fp64 of the same routed set: one token, tokens and blocks that fill no
tile, the largest block count, v stored either way, a gradient through the returned router
scores, frozen parameters, and the form that torch ops keep (a differentiated backward)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

CASES = [  # hidden, block, n_blocks, base, remote, tokens
    (64, 64, 2, 1, 1, 1),
    (64, 8, 17, 0, 5, 17),       # 17 blocks: one past a lane group
    (256, 16, 256, 4, 60, 33),   # most blocks; two (block, dim) accumulator sets
    (128, 64, 128, 128, 0, 15),  # every block, none routed
    (128, 32, 129, 2, 30, 5000), # several tiles of tokens per workgroup
]


def _module(fsi, case, dtype, dev, seed=0):
    D, bs, nb, base, remote, M = case
    torch.manual_seed(seed + sum(case))
    m = fsi.FovealPattentionMLP(hidden_dim=D, intermediate_dim=nb * bs, block_size=bs, base_blocks=base,
                                remote_blocks=remote, dtype=torch.float32)
    with torch.no_grad():
        m.block_keys_16d.normal_()
        m.out_proj_16d.weight.normal_(std=0.1)
    m = m.to(dev, dtype).train()
    x = torch.randn(M, D, device=dev).to(dtype)
    return m, x, torch.randn(M, D, device=dev).to(dtype)


def _reference(m, x, active, temperature=1.0):
    """(out, scores) in fp64 with autograd, for the given blocks."""
    w = {n: p.detach().double().requires_grad_() for n, p in m.named_parameters()}
    x = x.detach().double().requires_grad_()
    rows = (active.long()[:, None] * m.block_size + torch.arange(m.block_size, device=active.device)).flatten()
    z = F.rms_norm(x @ w["q_proj_16d.weight"].t(), (16,), eps=torch.finfo(torch.float32).eps)
    s = z @ w["block_keys_16d"].t() / 4.0
    ctx = torch.softmax(s / temperature, -1) @ w["block_keys_16d"]
    y = (F.silu(x @ w["k_gate"][rows].t()) * (x @ w["k_up"][rows].t())) @ w["v"][rows]
    return y + ctx @ w["out_proj_16d.weight"].t(), s, x, w


def _close(a, b, tol):
    b = b.double()
    return (a.double() - b).norm() <= tol * b.norm().clamp_min(1e-12)


# fp32: sums of up to 5000 products; bf16: each stored intermediate rounds to 2^-9 relative,
# and five of them lie on the router's path
TOL = {torch.float32: 2e-5, torch.bfloat16: 2.5e-2}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[f"k{i}" for i in range(len(CASES))])
def test_training_kernels(fsi, dev, case, dtype):
    print(f"[case] mlp training {case} {dtype}", flush=True)
    m, x, dy = _module(fsi, case, dtype, dev)
    nb, base, remote = case[2:5]
    xg = x.clone().requires_grad_()
    out, info = m(xg, return_router_info=True)
    assert m._train_fused(x)
    active = info["active_blocks"]
    assert active.dtype == torch.int32 and active[:base].tolist() == list(range(base))
    assert len(set(active.tolist())) == base + remote and int(active.max()) < nb
    mean = info["scores"].detach().mean(0)[base:].float()
    if remote:
        chosen = torch.zeros(nb - base, dtype=torch.bool, device=dev)
        chosen[active[base:].long() - base] = True
        if not bool(chosen.all()):
            assert mean[chosen].min() >= mean[~chosen].max()
    ds = torch.randn_like(info["scores"]) * 0.01
    torch.autograd.backward((out, info["scores"]), (dy, ds))
    ref, s, xr, w = _reference(m, x, active)
    torch.autograd.backward((ref, s), (dy.double(), ds.double()))
    assert _close(info["scores"], s, TOL[dtype]) and _close(out, ref, TOL[dtype])
    assert _close(xg.grad, xr.grad, TOL[dtype])
    for n, p in m.named_parameters():
        assert p.grad.shape == p.shape and p.grad.dtype == dtype
        assert _close(p.grad, w[n].grad, TOL[dtype]), n


def test_training_forms(fsi, dev):
    """v stored row-major, frozen weights, gradients of some outputs only, create_graph and
    autocast give what the usual form gives."""
    case = (64, 16, 24, 2, 6, 40)
    m, x, dy = _module(fsi, case, torch.float32, dev)
    params = dict(m.named_parameters())

    def grads(names, **kw):
        out = m(x)
        return torch.autograd.grad(out, [params[n] for n in names], dy, **kw)

    names = list(params)
    base = dict(zip(names, grads(names)))
    for n, g in zip(names, grads(names, create_graph=True)):
        assert g.requires_grad and _close(g.detach(), base[n], 1e-5), n
    for n in names:
        params[n].requires_grad_(False)
    params["v"].requires_grad_(True)
    assert _close(grads(["v"])[0], base["v"], 1e-6)
    params["v"].requires_grad_(False)
    params["block_keys_16d"].requires_grad_(True)
    _, info = m(x, return_router_info=True)
    (g,) = torch.autograd.grad(info["scores"].sum(), [params["block_keys_16d"]])
    assert torch.isfinite(g).all()
    for n in names:
        params[n].requires_grad_(True)
    with torch.no_grad():
        m.v = torch.nn.Parameter(m.v.detach().contiguous())
    assert m.v.stride(1) == 1
    params = dict(m.named_parameters())
    for n, g in zip(names, grads(names)):
        assert _close(g, base[n], 1e-5), n
    with torch.autocast("cuda", torch.bfloat16):
        assert not m._train_fused(x)
        assert torch.isfinite(m(x)).all()


def test_training_nan_tokens_route_in_range(fsi, dev):
    """NaN scores still give distinct blocks in range."""
    m, x, _ = _module(fsi, (64, 16, 24, 2, 6, 40), torch.bfloat16, dev)
    x[3] = float("nan")
    _, info = m(x, return_router_info=True)
    active = info["active_blocks"].tolist()
    assert len(set(active)) == 8 and 0 <= min(active) and max(active) < 24


def test_training_queries_of_another_type(fsi, dev):
    """A hook that widens the projected queries over bf16 keys is refused, as torch.matmul does."""
    m, x, _ = _module(fsi, (64, 16, 24, 2, 6, 40), torch.bfloat16, dev)
    m.q_proj_16d.register_forward_hook(lambda mod, a, out: out.float())
    with pytest.raises(RuntimeError):
        m(x)


def test_training_learnable_temperature(fsi, dev):
    """A temperature parameter gets the gradient of softmax(scores / T)."""
    m, x, dy = _module(fsi, (64, 16, 24, 2, 6, 40), torch.float32, dev)
    m.temperature = torch.nn.Parameter(torch.tensor(0.7, device=dev))
    out, info = m(x, return_router_info=True)
    (got,) = torch.autograd.grad(out, [m.temperature], dy)
    t = m.temperature.detach().double().requires_grad_()
    w = {n: p.detach() for n, p in m.named_parameters()}
    ref = torch.softmax(info["scores"].detach().double() / t, -1) @ w["block_keys_16d"].double()
    (want,) = torch.autograd.grad(ref @ w["out_proj_16d.weight"].double().t(), [t], dy.double())
    assert _close(got, want, 1e-4)


def test_training_softmax_tail(fsi, dev):
    """Single probabilities of the fp32 router softmax, read off a context of one-hot keys.
    Block 0 scores 2 z, blocks 1 .. 3 score -2 z, z and 0 with z of many values up to 4 sqrt(2), so
    every difference to the maximum is exact in fp32.  Bound: expf 2^-23 (one ulp), the sum of
    four terms and the quotient three roundings of 2^-24, the returned scores' own rounding none:
    3.0e-7."""
    m = fsi.FovealPattentionMLP(hidden_dim=64, intermediate_dim=64, block_size=16, base_blocks=1, remote_blocks=1,
                                dtype=torch.float32).to(dev).train()
    M = 2048
    q = torch.zeros(M, 16, device=dev)
    a = torch.linspace(0.0, 1.5, M, device=dev)
    q[:, 0], q[:, 1] = a.sin(), a.cos()
    keys = torch.zeros(4, 16, device=dev)
    keys[:, 0] = torch.tensor([8.0, -8.0, 4.0, 0.0], device=dev)
    keys[1, 5], keys[2, 6], keys[3, 7] = 1.0, 1.0, 1.0  # q is zero there
    s, ctx, _ = fsi.foveal_pattention._train_route_op(q, keys, 1, 1, 1.0)
    assert torch.equal(s[:, 1], -s[:, 0]) and torch.equal(2 * s[:, 2], s[:, 0]) and not s[:, 3].any()
    p = torch.softmax(s.double(), -1)[:, 1:]
    assert ((ctx[:, 5:8].double() - p) / p).abs().max() <= 3e-7
