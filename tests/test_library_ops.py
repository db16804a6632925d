"""torch.library registration (CPU only: FakeTensor tracing, no kernel runs).

Every HIP launch of the package is a custom op torch.ops.fsi.<name>; these tests
check that the expected ops exist, that their fake implementations give the
shapes and dtypes the real launches produce, and that a routed decode step
traces into a graph whose nodes are the fsi ops (what torch.compile / export
see)."""
import ctypes

import numpy as np
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

EXPECTED = {
    "additive_context", "additive_context_bwd", "block_scores", "block_scores_bwd", "block_sparse_linear",
    "blockwise_matmul", "decode_attention", "decode_route", "decode_step_attention", "dense_block_targets", "distill_kl", "distill_kl_bwd",
    "index_rms_norm", "index_rms_norm_bwd", "kv_page_pool", "kv_read", "kv_write", "masked_softmax",
    "masked_softmax_bwd", "mlp_router", "pattention", "pattention_pack", "pattention_packed", "pool_kv",
    "pool_kv_bwd", "route_from_scores", "score_and_route", "sparse_attention", "sram_indexer_attention", "swiglu",
    "swiglu_bwd", "tile_route",
}


@pytest.fixture(scope="module")
def ops(fsi):
    return torch.ops.fsi


def test_every_launch_is_registered(ops):
    have = {n for n in dir(ops) if not n.startswith("_") and n != "name"}
    assert EXPECTED <= have, EXPECTED - have


def _fake(*shape, dtype=torch.bfloat16):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def test_fake_shapes(ops):
    with FakeTensorMode():
        s = _fake(2, 8, 32, dtype=torch.float32)
        idx, cnt = ops.route_from_scores(s, True, 2, 0.9, 0, 4, 6, None, None, None, 0)
        assert idx.shape == (2, 8, 6) and idx.dtype == torch.int32 and cnt.shape == (2, 8)
        i2, c2, mass = ops.score_and_route(_fake(2, 5, 16), _fake(1, 40, 16), False, 0, 0.9, 0, 8, 8, True)
        assert i2.shape == (2, 5, 8) and mass.shape == (2, 5) and mass.dtype == torch.float32
        x = _fake(64, 4096)
        y = ops.pattention(x, _fake(14336, 4096), _fake(14336, 4096), _fake(14336, 4096), _fake(64, dtype=torch.int32),
                           64, 0, 1, False)
        assert y.shape == (64, 4096) and y.dtype == torch.bfloat16
        y = ops.pattention_packed(x, _fake(1 << 20, dtype=torch.uint8), None, 14336, 4096, 64, 1)
        assert y.shape == (64, 4096)
        a, sc = ops.mlp_router(x, _fake(16, 4096), _fake(224, 16), 8, 56, 1.0, True)
        assert a.shape == (64,) and a.dtype == torch.int32 and sc.shape == (224,)
        q = _fake(2, 8, 256, 64)
        kv = _fake(2, 2, 256, 64)
        o = ops.sparse_attention(q, kv, kv, _fake(2, 4, 3, dtype=torch.int32), _fake(2, 4, dtype=torch.int32), 3, 64,
                                 0, 64, 0.125)
        assert o.shape == q.shape and o.transpose(1, 2).is_contiguous()
        pages, counts, ctx = ops.decode_route(_fake(4, 16), _fake(4, 10, 16, dtype=torch.float32), _fake(4, 10, 16),
                                              None, 700, 64, 256, 10, 0.9, 2, 6, 6, True)
        assert pages.shape == (4, 6) and counts.shape == (4,) and ctx.shape == (4, 16)
        q3 = _fake(4, 8, 128)
        o = ops.decode_attention(q3, _fake(40, 2, 64, 128), _fake(40, 2, 64, 128), _fake(4, 10, dtype=torch.int32),
                                 10, 40, 640, 64, 2, None, 700, 256, None, None, 0, 0.1)
        assert o.shape == q3.shape
        lin = ops.block_sparse_linear(_fake(10, 256), _fake(512, 256), None, _fake(3, dtype=torch.int32), 64)
        assert lin.shape == (10, 512)
        mask, probs, need = ops.tile_route(_fake(7, 48, dtype=torch.float32), 0.5, 2, 3)
        assert mask.shape == (3, 48) and mask.dtype == torch.uint8 and probs.shape == (7, 48) and need.shape == (7,)
        out, sel = ops.sram_indexer_attention(_fake(2, 4, 64, 32, dtype=torch.float16),
                                              _fake(2, 4, 64, 32, dtype=torch.float16),
                                              _fake(2, 4, 64, 32, dtype=torch.float16),
                                              _fake(2, 4, 16, dtype=torch.float16), _fake(2, 4, 16, dtype=torch.float16),
                                              0.17, 0.8, 2, 16, True)
        assert out.shape == (2, 4, 64, 32) and sel.shape == (2, 4, 2) and sel.dtype == torch.int32
        loss, n = ops.distill_kl(_fake(2, 4, 9, dtype=torch.float32), _fake(2, 4, 9, dtype=torch.float32), 0, None,
                                 1.0)
        assert loss.shape == () and n.shape == (1,)


def test_decode_step_traces_to_fsi_ops(fsi):
    """A routed decode step (router -> packed Pattention) traced with fake
    tensors: the graph's call nodes are the two fsi ops."""
    buf_bytes = 1 << 20

    def step(x, wq, keys, buf):
        active = torch.ops.fsi.mlp_router(x, wq, keys, 8, 56, 1.0, False)[0]
        return torch.ops.fsi.pattention_packed(x, buf, active, 14336, 4096, 64, 1)

    with FakeTensorMode():
        args = (_fake(64, 4096), _fake(16, 4096), _fake(224, 16), _fake(buf_bytes, dtype=torch.uint8))
        gm = make_fx(step, tracing_mode="fake")(*args)
    targets = [str(n.target) for n in gm.graph.nodes if n.op == "call_function"]
    assert any("fsi.mlp_router" in t for t in targets) and any("fsi.pattention_packed" in t for t in targets)


def test_plain_call_only_where_the_dispatcher_has_nothing_to_do(fsi):
    """A launch function is called past torch.ops only for plain tensors that autograd would
    not record, outside every tracing, mode and transform."""
    import torch.autograd.forward_ad as fwad
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode

    plain = fsi._lib._plain_call
    t = torch.zeros(3)
    leaf = torch.zeros(3, requires_grad=True)
    assert plain((t, 1, None, torch.nn.Parameter(t, requires_grad=False)))
    assert not plain((t, leaf))
    with torch.no_grad():
        assert plain((t, leaf))

    class Sub(torch.Tensor):
        pass

    assert not plain((t.as_subclass(Sub),))
    with FakeTensorMode() as mode:
        fake = mode.from_tensor(t)
        assert not plain((fake,))
    assert not plain((fake,))

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not plain((t,))
    with torch.overrides.TorchFunctionMode():
        assert not plain((t,))
    with fwad.dual_level():
        assert not plain((t,))
    seen = []
    torch.func.vmap(lambda a: (seen.append(plain((a,))), a)[1])(torch.zeros(2, 3))
    torch.func.grad(lambda a: (seen.append(plain((t,))), a.sum())[1])(t)
    assert seen == [False, False]


def _toy(fsi, name):
    """An op of the package's kind whose launch reads memory, as a kernel does."""
    @fsi._lib.fsi_op(name, lambda x, n, s: torch.empty_like(x))
    def launch(x: torch.Tensor, n: int, s: float) -> torch.Tensor:
        raw = (ctypes.c_float * x.numel()).from_address(x.data_ptr())
        return torch.tensor(list(raw)).view(x.shape) * (n * s)

    return launch


def test_negated_view_reaches_the_launch_materialised(fsi):
    """A contiguous view with the negative bit set: its memory holds the other sign."""
    t = torch.tensor([1.0, -2.0, 3.0])
    view = torch._neg_view(t)
    assert view.is_neg() and view.is_contiguous() and not fsi._lib._plain_call((view,))
    assert torch.equal(_toy(fsi, "toy_negated")(view, 1, 1.0), -t)


def test_batched_gradients_go_through_the_dispatcher(fsi):
    """torch.autograd.grad(is_grads_batched=True) calls a backward once with a tensor that
    stands for the batch and has no storage; the dispatcher splits it."""
    op = _toy(fsi, "toy_batched")

    class Fn(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return op(x, 2, 1.0)

        @staticmethod
        def backward(ctx, g):
            return op(g, 2, 1.0)

    x = torch.ones(3, requires_grad=True)
    (got,) = torch.autograd.grad(Fn.apply(x), x, torch.eye(3), is_grads_batched=True)
    assert torch.equal(got, 2 * torch.eye(3))


@pytest.mark.parametrize("n", [np.int64(3), np.int32(3), torch.tensor(3)], ids=["int64", "int32", "tensor"])
@pytest.mark.parametrize("s", [0.5, np.float32(0.5), torch.tensor(0.5)], ids=["float", "float32", "tensor"])
def test_scalars_are_converted(fsi, n, s):
    """A size or scale that is no Python number arrives at the launch (a ctypes call) as one."""
    seen = []

    @fsi._lib.fsi_op(f"toy_scalar_{type(n).__name__}_{type(s).__name__}", lambda x, n, s: torch.empty_like(x))
    def launch(x: torch.Tensor, n: int, s: float) -> torch.Tensor:
        seen.append((type(n), type(s), n, s))
        return x * 2

    launch(torch.ones(2), n, s)
    assert seen == [(int, float, 3, 0.5)]


def test_numbers_of_the_other_kind(fsi):
    """What a schema refuses stays refused, and a whole number is a float where one is wanted."""
    op = _toy(fsi, "toy_other")
    with pytest.raises((RuntimeError, TypeError)):
        op(torch.ones(2), 3.0, 1.0)
    assert op(torch.ones(2), 2, 1).tolist() == [2.0, 2.0]


def test_every_launch_annotates_its_arguments(fsi):
    plain = {torch.Tensor, torch.nn.Parameter, int, float, bool, str, type(None)}
    for name in ("attention", "block_matmul", "core", "foveal_pattention", "pattention"):
        for f in vars(getattr(fsi, name)).values():
            if hasattr(f, "op") and hasattr(f, "__wrapped__"):
                kinds = fsi._lib._argument_kinds(f.__wrapped__)
                assert len(kinds) == f.__wrapped__.__code__.co_argcount and all(k <= plain for k in kinds), f


def test_keyword_arguments(fsi):
    assert _toy(fsi, "toy_keyword")(torch.ones(2), s=0.5, n=4).tolist() == [2.0, 2.0]


def test_profiler_lists_the_ops(fsi):
    op = _toy(fsi, "toy_profiled")
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        op(torch.ones(2), 1, 1.0)
    assert "fsi::toy_profiled" in {e.key for e in prof.key_averages()}
