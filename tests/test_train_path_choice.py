"""Which FovealPattentionMLP training calls the fused kernels take (CPU only: FakeTensor
tracing of the forward, no kernel runs).  Whatever the module's owner puts in the place of a
part that the fused path would pass by keeps the torch form, which calls it."""
import pytest
import torch
from torch import nn
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode


class _Ops(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def _traced(fsi, change=None, dtype=torch.bfloat16):
    """Names of the ops of one training forward after change(module)."""
    with FakeTensorMode(), torch.device("cuda"):
        m = fsi.FovealPattentionMLP(hidden_dim=256, intermediate_dim=1024, base_blocks=2, remote_blocks=4,
                                    dtype=dtype).train()
        if change is not None:
            change(m)
        with _Ops() as ops:
            m(torch.empty(2, 8, 256, dtype=dtype))
    return ops.names


def _fused(names):
    return any("fsi.mlp_train_route" in n for n in names)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_plain_module_is_fused(fsi, dtype):
    assert _fused(_traced(fsi, dtype=dtype))


def test_hooked_projection_keeps_torch_ops(fsi):
    """A hook that returns fp32 queries over bf16 keys: torch.matmul decides on the pair; the
    kernel would read the keys as fp32, past their end."""
    assert not _fused(_traced(fsi, lambda m: m.q_proj_16d.register_forward_hook(lambda mod, a, out: out.float())))


def test_route_op_refuses_mixed_operands(fsi):
    route, bwd = fsi.foveal_pattention._train_route_op, fsi.foveal_pattention._train_route_bwd_op
    q, keys = torch.zeros(3, 16), torch.zeros(4, 16)
    for args in ((q, keys.bfloat16()), (q.bfloat16(), keys)):
        with pytest.raises(TypeError, match="dtype mismatch"):
            route(*args, 1, 2, 1.0)
        with pytest.raises(TypeError, match="dtype mismatch"):
            bwd(*args, None, None, 1.0)
    for args in ((q[:, :8], keys), (q, keys[:, :8])):
        with pytest.raises(ValueError, match="rows of 16"):
            route(*args, 1, 2, 1.0)


class _Wrapped(nn.Module):
    """A projection without a weight of its own."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        return self.inner(x) * 2


def test_wrapped_projection_is_called(fsi):
    def wrap(m):
        m.q_proj_16d = _Wrapped(m.q_proj_16d)

    assert not _fused(_traced(fsi, wrap))


def _biased(self, x):
    self.calls = getattr(self, "calls", 0) + 1
    return torch.matmul(self.q_proj_16d(x), self.block_keys_16d.t()) + 1.0


@pytest.mark.parametrize("where", ["subclass", "instance", "class"])
def test_replaced_router_scores_are_called(fsi, where, monkeypatch):
    """compute_router_scores is what the training forward routes on, whoever replaced it."""
    seen = []

    def change(m):
        if where == "subclass":
            m.__class__ = type("Biased", (fsi.FovealPattentionMLP,), {"compute_router_scores": _biased})
        elif where == "instance":
            m.compute_router_scores = _biased.__get__(m)
        else:
            monkeypatch.setattr(fsi.FovealPattentionMLP, "compute_router_scores", _biased)
        seen.append(m)

    assert not _fused(_traced(fsi, change))
    assert seen[0].calls == 1


@pytest.mark.parametrize("temperature", ["parameter", "tensor", 0.0, -1.0, 1e-50, float("inf"), float("nan")])
def test_temperature_keeps_torch_ops(fsi, temperature):
    """A learnable or tensor temperature has its gradient through scores / temperature; numbers
    whose reciprocal fp32 does not hold divide in torch."""
    def change(m):
        if temperature == "parameter":
            m.temperature = nn.Parameter(torch.ones(()))
        elif temperature == "tensor":
            m.temperature = torch.ones((), requires_grad=True)
        else:
            m.temperature = temperature

    assert not _fused(_traced(fsi, change))


@pytest.mark.parametrize("temperature", [1, 0.5])
def test_number_temperature_is_fused(fsi, temperature):
    assert _fused(_traced(fsi, lambda m: setattr(m, "temperature", temperature)))


@pytest.mark.parametrize("name", ["k_gate", "k_up", "v"])
def test_weights_of_another_size_keep_torch_ops(fsi, name):
    """A shorter weight has no rows for some active blocks: indexing it is refused or not by
    torch; the gather kernel would read past its end."""
    def shorten(m):
        setattr(m, name, nn.Parameter(getattr(m, name).detach()[:512]))

    assert not _fused(_traced(fsi, shorten))


def test_gather_op_refuses_weights_of_two_sizes_or_types(fsi):
    w, active = torch.zeros(64, 16), torch.zeros(1, dtype=torch.int32)
    for ws in ((w, w[:32], w), (w, w, w[:32]), (w, w.bfloat16(), w)):
        with pytest.raises(ValueError, match="weights"):
            fsi.foveal_pattention._train_gather_op(*ws, active, 16, False)


class _Stored(torch.Tensor):
    """A weight in a storage form of its own (quantised, sharded) that indexing decodes."""

    @staticmethod
    def __new__(cls, like):
        return torch.Tensor._make_wrapper_subclass(cls, like.shape, dtype=like.dtype, device=like.device)

    def __init__(self, like):
        self.inner = like

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        args = [a.inner if isinstance(a, _Stored) else a for a in args]
        if func not in (torch.ops.aten.index.Tensor, torch.ops.aten.detach.default):
            raise NotImplementedError(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("name", ["k_gate", "k_up", "v"])
def test_weight_of_a_tensor_class_is_indexed(fsi, name):
    def store(m):
        w = getattr(m, name).detach()
        del m._parameters[name]
        setattr(m, name, _Stored(w))

    assert not _fused(_traced(fsi, store))
