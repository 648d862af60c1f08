"""The layer at few rows per expert, where its forward streams the routed and the shared experts'
weights in two launches (zmoe_glu_stream_shared_ok): against the oracle with its backward, and what the
route owes its callers."""

import pytest
import torch

from helpers import assert_close, gen, np64

pytestmark = pytest.mark.gpu


def _streams(T, d, f, fs, E, k):
    from zmoe import library as zl

    return zl.glu_stream_shared_ok(T, d, f, fs, E, k) and zl.glu_stream_shared_pays(T, d, fs)


def _layer(dev, dtype, d=128, E=64, k=4, f=64, n_shared=1, seed=0):
    from modeling.model_config import ModelConfig
    from modeling.moe_layer import MoELayer

    torch.manual_seed(seed)
    cfg = ModelConfig(hidden_size=d, intermediate_size=f, n_experts=E + n_shared, n_shared_experts=n_shared,
                      n_experts_per_token=k)
    layer = MoELayer(cfg).to(dev).to(dtype)
    layer.gate.expert_biases.data = (0.1 * torch.randn(E)).to(dev)
    return layer


def _step(layer, x, dout, between=None, autocast=False, **kw):
    """(out, dx, weight grads by name) of one step; ``between`` runs after the forward."""
    layer.zero_grad(set_to_none=True)
    x = x.clone().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        out, idx = layer(x, **kw)
    if between is not None:
        with torch.no_grad():
            between()
    out.backward(dout)
    return out.detach(), x.grad, {n: p.grad.clone() for n, p in layer.named_parameters()}


def _equal(a, b):
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for n in a[2]:
        assert torch.equal(a[2][n], b[2][n]), n


@pytest.mark.parametrize("T,n_shared", [(1, 1), (16, 1), (33, 2), (128, 2)])   # one to four groups of 32 tokens
def test_layer_against_oracle(hip_device, T, n_shared):
    """Forward and backward on the streaming route (bf16), every grad."""
    from test_gpu_layer import run_and_compare

    d, E, k, f = 128, 64, 4, 64
    assert _streams(T, d, f, n_shared * f, E, k)
    run_and_compare(T, d, E, k, f, n_shared, torch.bfloat16, hip_device)


@pytest.mark.parametrize("pad", [False, True])
@pytest.mark.parametrize("T", [16, 33])
def test_fp32_masters_match_bf16_layer(hip_device, T, pad):
    """fp32 weights and input under bf16 autocast on the streaming route, with and without unpad
    indices: the bf16 layer's output bit for bit, its input grad's fp32 sum, and fp32 weight grads
    that round to its own but for rare accumulation flips (the bf16 layer itself: the oracle, above)."""
    l32, l16 = _layer(hip_device, torch.float32), _layer(hip_device, torch.float32)
    l16.load_state_dict(l32.state_dict())
    bias = l32.gate.expert_biases.data.clone()
    l16 = l16.to(torch.bfloat16)
    l16.gate.expert_biases.data = bias
    kw, n = {}, T
    if pad:
        kw["unpad_indices"] = torch.tensor([i for i in range(T) if i % 5 != 2], device=hip_device)
        n = kw["unpad_indices"].numel()
    assert _streams(n, 128, 64, 64, 64, 4)
    x = torch.randn(1, T, 128, generator=gen(6)).to(torch.bfloat16).to(hip_device)
    dout = torch.randn(1, T, 128, generator=gen(7)).to(torch.bfloat16).to(hip_device)
    o32, dx32, g32 = _step(l32, x.float(), dout, autocast=True, **kw)
    o16, dx16, g16 = _step(l16, x, dout, **kw)
    assert torch.equal(o32, o16)
    assert dx32.dtype == torch.float32 and torch.equal(dx32.to(torch.bfloat16), dx16)
    for name, g in g32.items():
        r = g.to(torch.bfloat16)
        assert g.dtype == torch.float32 and g16[name].abs().sum() > 0, name
        assert (r == g16[name]).float().mean().item() >= 0.99, name
        assert_close(np64(r), np64(g16[name]), rtol=2 ** -7, atol=1e-6, what=name)


def test_weights_edited_between_forward_and_backward(hip_device):
    """The backward takes the shared expert's up and gate and the router as the forward saw them."""
    T, dt = 16, torch.bfloat16
    assert _streams(T, 128, 64, 64, 64, 4)
    layer = _layer(hip_device, dt)
    x = torch.randn(1, T, 128, generator=gen(1)).to(dt).to(hip_device)
    dout = torch.randn(1, T, 128, generator=gen(2)).to(dt).to(hip_device)
    ref = _step(layer, x, dout)
    se = layer.shared_experts
    _equal(_step(layer, x, dout, lambda: [w.mul_(2) for w in (layer.gate.weight, se.up_proj.weight,
                                                              se.gate_proj.weight)]), ref)


def _off16(layer, names):
    """The named weights as parameters that start one element into a buffer of their own."""
    for n in names:
        mod = layer.get_submodule(n.rpartition(".")[0])
        w = mod.weight.detach()
        buf = torch.empty(w.numel() + 1, dtype=w.dtype, device=w.device)
        view = buf[1:].view(w.shape)
        view.copy_(w)
        mod.weight = torch.nn.Parameter(view)
        assert mod.weight.data_ptr() % 16


SHARED = tuple(f"shared_experts.{p}_proj.weight" for p in ("up", "gate", "down"))


def test_shared_weights_off_16_bytes(hip_device):
    """A shared expert whose weights are views into a flat buffer: taken, with the same bits; the
    routed experts' weights are still refused there, as they are at every size."""
    T, dt = 8, torch.bfloat16
    assert _streams(T, 128, 64, 64, 64, 4)
    x = torch.randn(1, T, 128, generator=gen(3)).to(dt).to(hip_device)
    layer = _layer(hip_device, dt).requires_grad_(False)
    ref = layer(x)[0]
    for names in (SHARED[:1], SHARED[1:2], SHARED[2:], SHARED):
        layer = _layer(hip_device, dt).requires_grad_(False)
        _off16(layer, names)
        assert torch.equal(layer(x)[0], ref)
    _off16(layer, ("routed_experts.experts.weight",))
    with pytest.raises(ValueError):
        layer(x)


@pytest.mark.parametrize("T", [16, 300])   # the streaming route, and the other
def test_fp32_shared_weights_off_16_bytes(hip_device, T):
    """fp32 weights under bf16 autocast: the dense ones (shared expert, router) may start at any
    element, in the forward and the backward; the routed experts' are refused, as they always were."""
    assert _streams(T, 128, 64, 64, 64, 4) == (T == 16)
    x = torch.randn(1, T, 128, generator=gen(4)).to(hip_device)
    dout = torch.randn(1, T, 128, generator=gen(5)).to(torch.bfloat16).to(hip_device)
    ref = _step(_layer(hip_device, torch.float32), x, dout, autocast=True)
    for names in (SHARED[2:], ("gate.weight",), (*SHARED, "gate.weight")):
        layer = _layer(hip_device, torch.float32)
        _off16(layer, names)
        _equal(_step(layer, x, dout, autocast=True), ref)
    for name in ("routed_experts.experts.weight", "routed_experts.output_experts.weight"):
        layer = _layer(hip_device, torch.float32)
        _off16(layer, (name,))
        with pytest.raises(ValueError):
            _step(layer, x, dout, autocast=True)


@pytest.mark.parametrize("T", [192, 193])
def test_shared_expert_leaves_the_launches(hip_device, T, monkeypatch):
    """Few rows per routed expert, but so many tokens that the shared expert is better off in library
    GEMMs: the layer takes those (d = 2048, a shared width of 1536: from seven groups of 32 tokens)."""
    from test_gpu_layer import run_and_compare
    from zmoe import library as zl

    calls = []
    real = zl.glu_shared_forward
    monkeypatch.setattr(zl, "glu_shared_forward", lambda *a: calls.append(1) or real(*a))
    assert T * 1 <= 8 * 32
    run_and_compare(T, 2048, 32, 1, 64, 24, torch.bfloat16, hip_device)
    assert len(calls) == (T == 192)


def test_compiled_step_equals_eager(hip_device):
    """The streaming route under torch.compile with dynamic shapes, at two token counts, and at a third
    that leaves it."""
    import torch._dynamo

    layer = _layer(hip_device, torch.bfloat16)
    torch._dynamo.reset()
    fn = torch.compile(lambda x: layer(x), backend="aot_eager", dynamic=True, fullgraph=True)
    for T in (16, 33, 300):
        assert _streams(T, 128, 64, 64, 64, 4) == (T < 300)
        x = torch.randn(1, T, 128, generator=gen(T)).to(torch.bfloat16).to(hip_device)
        dout = torch.randn(1, T, 128, generator=gen(T + 1)).to(torch.bfloat16).to(hip_device)
        ref = _step(layer, x, dout)
        xg = x.clone().requires_grad_(True)
        layer.zero_grad(set_to_none=True)
        out, _ = fn(xg)
        out.backward(dout)
        _equal((out.detach(), xg.grad, {n: p.grad for n, p in layer.named_parameters()}), ref)
    torch._dynamo.reset()
