"""Host side of the 16-D index products (CPU only): second derivatives (the kernels' ops stand
in as the torch products that they compute, in fp64; linear layers, which they replace, can
be differentiated twice) and the rows that the kernels are handed."""
import pytest
import torch


@pytest.fixture
def core(fsi, monkeypatch):
    c = fsi.core

    def proj(x, w0, w1):
        return x @ w0.t(), x @ w1.t() if w1 is not None else x.new_empty((0,))

    def proj_dw(x, g0, g1):
        d = lambda g: g.reshape(-1, 16).t() @ x.reshape(-1, x.shape[-1])  # noqa: E731
        return d(g0), d(g1) if g1 is not None else x.new_empty((0,))

    def expand_bwd(dy, context, w, block):
        s = dy.reshape(*context.shape[:2], block, -1).sum(2)
        return s @ w, s.flatten(0, 1).t() @ context.flatten(0, 1)

    monkeypatch.setattr(c, "_proj_op", proj)
    monkeypatch.setattr(c, "_proj_dw_op", proj_dw)
    monkeypatch.setattr(c, "_expand_op", lambda ctx, w, n: (ctx @ w.t()).repeat_interleave(n, dim=1))
    monkeypatch.setattr(c, "_expand_bwd_op", expand_bwd)
    return c


def _leaves(*shapes):
    g = torch.Generator().manual_seed(0)
    return [torch.randn(*s, generator=g, dtype=torch.float64).requires_grad_() for s in shapes]


def test_projection_twice(core):
    x, w0, w1 = _leaves((2, 3, 5), (16, 5), (16, 5))
    both = lambda *a: core._Proj16Fn.apply(*a)  # noqa: E731
    one = lambda x, w: core._Proj16Fn.apply(x, w, None)[0]  # noqa: E731
    assert torch.autograd.gradcheck(both, (x, w0, w1)) and torch.autograd.gradgradcheck(both, (x, w0, w1))
    assert torch.autograd.gradcheck(one, (x[0], w0)) and torch.autograd.gradgradcheck(one, (x[0], w0))


def test_projection_gradient_of_one_output(core):
    """The input's gradient from a constant incoming gradient keeps its graph."""
    x, w0, w1 = _leaves((2, 3, 5), (16, 5), (16, 5))
    (dx,) = torch.autograd.grad(core._Proj16Fn.apply(x, w0, w1)[1].sum(), x, create_graph=True)
    assert torch.equal(torch.autograd.grad(dx.sum(), w1)[0], torch.full((16, 5), 6.0, dtype=torch.float64))


def test_expansion_twice(core):
    ctx, w = _leaves((2, 3, 16), (7, 16))
    f = lambda c, w: core._Expand16Fn.apply(c, w, 4)  # noqa: E731
    assert torch.autograd.gradcheck(f, (ctx, w)) and torch.autograd.gradgradcheck(f, (ctx, w))


ROWS = {  # shape, strides, first element
    "row": ((1, 1, 128), (130, 130, 1), 0),  # one row of a padded buffer
    "row2d": ((1, 128), (130, 1), 0),
    "batch": ((1, 4, 128), (516, 128, 1), 0),
    "rows of one": ((3, 1, 128), (136, 130, 1), 0),
    "odd rows": ((1, 4, 128), (520, 130, 1), 0),
    "odd start": ((1, 4, 128), (512, 128, 1), 1),
    "odd row start": ((1, 1, 128), (130, 130, 1), 1),
    "expanded": ((3, 4, 128), (0, 128, 1), 0),
    "turned": ((1, 4, 128), (512, 1, 4), 0),
}


@pytest.mark.parametrize("kind", ROWS)
def test_rows_are_aligned(fsi, kind):
    """What the kernels ask for: strides of whole 16-byte pieces, also where a dimension has one
    entry and torch leaves its stride as it was, and the same values at them."""
    x = torch.arange(1040).bfloat16().as_strided(*ROWS[kind])
    y, xs_b, xs_t = fsi.core._rows_3d(x)
    B, T, D = y.shape
    assert xs_b % 8 == 0 and xs_t % 8 == 0 and y.data_ptr() % 16 == 0 and y.stride(2) == 1
    assert torch.equal(y.as_strided((B, T, D), (xs_b, xs_t, 1), y.storage_offset()), x.reshape(B, T, D))


def test_ops_refuse_operands_of_other_shapes(fsi):
    """The kernels read 16 columns, or 16 components a row, of one type, whatever the memory holds."""
    core, z = fsi.core, torch.zeros
    x, w, c = z(2, 3, 128), z(16, 128), z(2, 3, 16)
    for call in (lambda: core._proj_op(x, w[:, :64], None), lambda: core._proj_op(x, w[:8], None),
                 lambda: core._proj_op(x, w, w[:8]), lambda: core._proj_dw_op(x, c[:, :2], None),
                 lambda: core._proj_dw_op(x, c, c[..., :8]), lambda: core._expand_op(c, z(16, 8), 4),
                 lambda: core._expand_op(c[..., :8], z(16, 8), 4),
                 lambda: core._expand_bwd_op(z(2, 12, 8), c, z(16, 16), 4),
                 lambda: core._expand_bwd_op(z(2, 6, 16), c, z(16, 16), 4)):
        with pytest.raises(ValueError):
            call()
    for call in (lambda: core._proj_op(x, w, w.bfloat16()), lambda: core._proj_dw_op(x, c.bfloat16(), None),
                 lambda: core._expand_op(c, z(16, 16).bfloat16(), 4)):
        with pytest.raises(TypeError, match="dtype mismatch"):
            call()


@pytest.mark.parametrize("shape", [(16, 8), (24, 16)])
def test_stream_of_a_replaced_out_proj(fsi, shape):
    """A projection of another input width is refused, as by the linear layer itself; 16 outputs
    are not 16 inputs."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode(), torch.device("cuda"):
        m = fsi.FovealIndexer(hidden_size=128, block_size=8)
        m.out_proj = torch.nn.Linear(shape[1], shape[0], bias=False)
        s, v = torch.empty(1, 2, 2), torch.empty(1, 2, 16)
        if shape[1] == 16:
            assert m.additive_stream(s, v).shape == (1, 16, 24)
        else:
            with pytest.raises(RuntimeError):
                m.additive_stream(s, v)
