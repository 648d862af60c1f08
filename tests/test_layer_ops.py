"""What sees the layer's ops (zmoe.library.layer_op): they are custom ops, and whatever watches a call or
has rules registered on an op meets it under its zmoe:: name; the native form runs for the rest."""

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode


class _Dispatched(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


class _Called(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


class _Wrapped(torch.Tensor):
    names = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.names.append(str(func))
        return super().__torch_function__(func, types, args, kwargs or {})


def _fake_cuda(*shape):
    return torch.empty(*shape, device="cuda", dtype=torch.bfloat16)


def test_ops_are_custom_ops():
    from scattermoe.kernels import ops as ko
    from zmoe import library as zl

    for op in (zl.combine, zl.grouped_mm, ko.scatter2scatter_compileable, ko.group_compileable):
        assert isinstance(op, torch.library.CustomOpDef)


def test_modes_and_graphs_hold_the_zmoe_names():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from zmoe import library as zl

    with FakeTensorMode(), torch.no_grad():
        H = _fake_cuda(4, 16)
        with _Dispatched() as seen:
            assert zl.swiglu(H).shape == (4, 8)
        assert seen.names == ["zmoe.swiglu.default"]
        graph = make_fx(lambda h: zl.swiglu(h))(H).graph
    assert torch.ops.zmoe.swiglu.default in [n.target for n in graph.nodes]


@pytest.fixture(scope="module")
def toy():
    """An op whose custom form doubles and whose native form triples."""
    from zmoe.library import layer_op

    @layer_op("toy_for_tests")
    def op(x: torch.Tensor) -> torch.Tensor:
        return 2 * x

    op.register_fake(lambda x: torch.empty_like(x))
    op.register_vmap(lambda info, in_dims, x: (5 * x, in_dims[0]))
    op._native = lambda x: 3 * x
    yield op
    torch._dynamo.reset()


def test_native_form_runs_unobserved_only(toy):
    x = torch.ones(3)
    assert torch.equal(toy(x), 2 * x)                      # grad mode on
    with torch.no_grad():
        assert torch.equal(toy(x), 3 * x)
        assert torch.equal(toy(torch.nn.Parameter(x)), 3 * x)
        with torch.device("cpu"):                          # a default device watches nothing
            assert torch.equal(toy(x), 3 * x)
        with _Dispatched() as seen:
            assert torch.equal(toy(x), 2 * x)
        assert "zmoe.toy_for_tests.default" in seen.names
        with _Called() as seen:
            assert torch.equal(toy(x), 2 * x)
        assert any("toy_for_tests" in n for n in seen.names)
        assert torch.equal(toy(x.as_subclass(_Wrapped)).as_subclass(torch.Tensor), 2 * x)
        assert any("toy_for_tests" in n for n in _Wrapped.names)
        assert torch.equal(torch.func.vmap(toy)(torch.ones(2, 3)), 5 * torch.ones(2, 3))  # the registered rule
        with torch.autograd.forward_ad.dual_level():
            assert torch.equal(toy(x), 2 * x)
        assert torch.equal(torch.compile(lambda v: toy(v), backend="eager", fullgraph=True)(x), 2 * x)
        assert torch.equal(toy(x), 3 * x)
    with torch.inference_mode():
        assert torch.equal(toy(x), 3 * x)


@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_jit_trace_records_the_zmoe_op(toy):
    with torch.no_grad():
        graph = torch.jit.trace(lambda v: toy(v), torch.ones(3), check_trace=False).graph
    assert "zmoe::toy_for_tests" in str(graph)
