"""The 16-D index's products on csrc/index_proj.hip (projections, their weight gradients, the
additive stream's expansion) against fp64: one row, rows that fill no tile, the switch between
its two tile shapes, strided rows, and the linear layers' own GEMMs where it does not apply."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float32]
# fp32: sums of up to 8200 products; bf16: one rounding of an fp32 sum
TOL = {torch.float32: 3e-6, torch.bfloat16: 3e-3}


def _close(a, b, dtype):
    return (a.double() - b).norm() <= TOL[dtype] * b.norm().clamp_min(1e-30)


@pytest.mark.parametrize("dtype", DTYPES, ids=["bf16", "f32"])
@pytest.mark.parametrize("B,T,D,step", [(1, 1, 128, 1), (1, 17, 256, 1), (2, 65, 128, 1), (3, 100, 1024, 7),
                                        (1, 8191, 128, 1), (2, 4100, 256, 1), (2, 8200, 128, 2)])
def test_projection_and_weight_gradient(fsi, dev, dtype, B, T, D, step):
    print(f"[case] projection B={B} T={T} D={D} step={step} {dtype}", flush=True)
    g = torch.Generator().manual_seed(B + T + D)
    full = torch.randn(B, T, D, generator=g).to(dev, dtype)
    x = full[:, ::step]
    if step == 7:
        x = x[:, 1:]  # rows no multiple of a batch entry
    w = [torch.randn(16, D, generator=g).to(dev, dtype) for _ in range(2)]
    dy = [torch.randn(*x.shape[:2], 16, generator=g).to(dev, dtype) for _ in range(2)]
    core = fsi.core
    for n in (1, 2):
        y = core._proj_op(x, w[0], w[1] if n == 2 else None)
        dw = core._proj_dw_op(x, dy[0], dy[1] if n == 2 else None)
        x2 = x.reshape(-1, D).double()
        for i in range(n):
            assert _close(y[i], x.double() @ w[i].double().t(), dtype)
            assert _close(dw[i], dy[i].reshape(-1, 16).double().t() @ x2, dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=["bf16", "f32"])
@pytest.mark.parametrize("B,nb,block,D", [(1, 1, 1, 8), (2, 3, 16, 64), (1, 40, 64, 2056), (1, 9, 5, 4104)])
def test_expansion(fsi, dev, dtype, B, nb, block, D):
    print(f"[case] expansion B={B} nb={nb} block={block} D={D} {dtype}", flush=True)
    g = torch.Generator().manual_seed(nb + D)
    c, w = torch.randn(B, nb, 16, generator=g).to(dev, dtype), torch.randn(D, 16, generator=g).to(dev, dtype)
    dy = torch.randn(B, nb * block, D, generator=g).to(dev, dtype)
    core = fsi.core
    out = core._expand_op(c, w, block)
    assert _close(out, (c.double() @ w.double().t()).repeat_interleave(block, 1), dtype)
    dc, dw = core._expand_bwd_op(dy, c, w, block)
    s = dy.double().view(B, nb, block, D).sum(2)
    assert _close(dc, s @ w.double(), dtype)
    assert _close(dw, s.reshape(-1, D).t() @ c.reshape(-1, 16).double(), dtype)


def test_expansion_backward_keeps_no_scratch(fsi, dev):
    """With blocks of one element the block sums are as large as the gradient itself."""
    c, w = torch.randn(2, 2000, 16, device=dev), torch.randn(2048, 16, device=dev)
    kept = lambda: sum(b.numel() for b in fsi._lib._ws.values())  # noqa: E731
    before = kept()
    fsi.core._expand_bwd_op(torch.randn(2, 2000, 2048, device=dev), c, w, 1)
    assert kept() == before


@pytest.mark.parametrize("why", ["plain", "hook", "bias", "width", "autocast", "odd"])
def test_indexer_paths_agree(fsi, dev, why):
    """The indexer's representations and gradients are those of its linear layers, whichever
    way they run; a hook, a bias or autocast keeps the layers themselves."""
    D = 96 if why == "width" else 128
    torch.manual_seed(0)
    m = fsi.FovealIndexer(hidden_size=D, block_size=8).to(dev)
    with torch.no_grad():
        m.out_proj.weight.normal_()
    calls = []
    if why == "hook":
        for lin in (m.q_proj, m.k_proj, m.v_proj, m.out_proj):
            lin.register_forward_hook(lambda *a: calls.append(1))
    if why == "bias":
        for lin in (m.q_proj, m.k_proj, m.v_proj):
            lin.bias = torch.nn.Parameter(torch.zeros(16, device=dev))
    x = torch.randn(2, 40, D + 1, device=dev)[..., 1:] if why == "odd" else torch.randn(2, 40, D, device=dev)
    x.requires_grad_()

    def run(mod, x, f=lambda t: t):
        import torch.nn.functional as F
        q = F.rms_norm(f(x) @ f(mod.q_proj.weight).t(), (16,), eps=torch.finfo(torch.float32).eps)
        k = F.rms_norm(f(x) @ f(mod.k_proj.weight).t(), (16,), eps=torch.finfo(torch.float32).eps)
        k = F.normalize(k.view(2, 5, 8, 16).mean(2), dim=-1)
        v = (f(x) @ f(mod.v_proj.weight).t()).view(2, 5, 8, 16).mean(2)
        return q, k, v

    if why == "autocast":
        with torch.autocast("cuda", torch.bfloat16):
            assert m.compute_query_16d(x).dtype == torch.bfloat16
        return
    q, (k, v) = m.compute_query_16d(x), m.compute_kv_blocks_16d(x)
    qr, kr, vr = run(m, x, lambda t: t.double())
    for a, b in ((q, qr), (k, kr), (v, vr)):
        assert _close(a.detach(), b.detach(), torch.float32)
    dq, dk, dv = (torch.randn_like(t) for t in (q, k, v))
    leaves = [x, m.q_proj.weight, m.k_proj.weight, m.v_proj.weight]
    got = torch.autograd.grad((q, k, v), leaves, (dq, dk, dv))
    want = torch.autograd.grad((qr, kr, vr), leaves, (dq.double(), dk.double(), dv.double()))
    for a, b in zip(got, want):
        assert (a.double() - b).norm() <= 1e-5 * b.double().norm()
    s, vv = torch.randn(2, 5, 5, device=dev, requires_grad=True), v.detach().requires_grad_()
    valid = torch.arange(5, device=dev)[None] < torch.arange(5, device=dev)[:, None]
    add = m.additive_stream(s, vv)
    sd, vd, wd = (t.detach().double().requires_grad_() for t in (s, vv, m.out_proj.weight))
    p = torch.nan_to_num(torch.softmax(sd.masked_fill(~valid, float("-inf")), -1))
    ref = ((p @ vd) @ wd.t()).repeat_interleave(8, dim=1)
    assert add.shape == (2, 40, D) and _close(add.detach(), ref.detach(), torch.float32)
    dy = torch.randn_like(add)
    for a, b in zip(torch.autograd.grad(add, (s, vv, m.out_proj.weight), dy),
                    torch.autograd.grad(ref, (sd, vd, wd), dy.double())):
        assert b.any() and (a.double() - b).norm() <= 1e-5 * b.norm()
    assert len(calls) == (4 if why == "hook" else 0)


def test_additive_stream_second_derivative(fsi, dev):
    """A penalty on out_proj's gradient reaches the scores and values, as through nn.Linear."""
    torch.manual_seed(3)
    m = fsi.FovealIndexer(hidden_size=128, block_size=8).to(dev)
    with torch.no_grad():
        m.out_proj.weight.normal_()
    s, v = torch.randn(2, 5, 5, device=dev, requires_grad=True), torch.randn(2, 5, 16, device=dev, requires_grad=True)
    dy = torch.randn(2, 40, 128, device=dev)

    def second(stream, s, v, w, dy):
        (dw,) = torch.autograd.grad(stream, w, dy, create_graph=True)
        return torch.autograd.grad(dw.square().sum(), (s, v))

    got = second(m.additive_stream(s, v), s, v, m.out_proj.weight, dy)
    sd, vd, wd = (t.detach().double().requires_grad_() for t in (s, v, m.out_proj.weight))
    valid = torch.arange(5, device=dev)[None] < torch.arange(5, device=dev)[:, None]
    p = torch.nan_to_num(torch.softmax(sd.masked_fill(~valid, float("-inf")), -1))
    ref = ((p @ vd) @ wd.t()).repeat_interleave(8, dim=1)
    for a, b in zip(got, second(ref, sd, vd, wd, dy.double())):
        assert b.any() and (a.double() - b).norm() <= 1e-5 * b.norm()


@pytest.mark.parametrize("shape,strides", [((1, 1, 128), (130, 130, 1)), ((1, 4, 128), (514, 128, 1)),
                                           ((3, 1, 128), (136, 130, 1))])
def test_one_row_or_sequence_of_a_padded_buffer(fsi, dev, shape, strides):
    """A dimension of one entry has a stride that no copy changes."""
    torch.manual_seed(0)
    m = fsi.FovealIndexer(hidden_size=128, block_size=1).to(dev)
    x = torch.randn(600, device=dev).as_strided(shape, strides)
    q, (k, v) = m.compute_query_16d(x), m.compute_kv_blocks_16d(x)
    weights = [m.q_proj.weight, m.k_proj.weight, m.v_proj.weight]
    dy = [torch.randn_like(t) for t in (q, k, v)]
    got = torch.autograd.grad((q, k, v), weights, dy)
    y = x.clone(memory_format=torch.contiguous_format)
    q2, (k2, v2) = m.compute_query_16d(y), m.compute_kv_blocks_16d(y)
    assert torch.equal(q, q2) and torch.equal(k, k2) and torch.equal(v, v2)
    for a, b in zip(got, torch.autograd.grad((q2, k2, v2), weights, dy)):
        assert torch.equal(a, b)
