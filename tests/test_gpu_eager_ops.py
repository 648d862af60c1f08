"""The native dispatcher kernels of the layer's ops (csrc/eager_ops.cpp, zmoe_eager::) against the
ops' general form (zmoe::, the Python wrappers): the same bits for the operands the layer passes,
for strided rows, other index and gate dtypes and widths that need padding, the same errors, and
the general form where a backward through the op has to be refused. That an op runs natively is shown
by taking the general form's functions away."""

import threading

import pytest
import torch

from helpers import gen

pytestmark = pytest.mark.gpu

T, K2, E, D, F = 37, 2, 8, 64, 40  # E a multiple of 8: swiglu_route_backward packs [2f + E] rows


def _ops(dev, dtype, d, f):
    """name -> (args, ...) for every op, at T tokens, K2 slots, E experts."""
    g = gen(d + f)
    r = lambda *s, dt=dtype: torch.randn(*s, generator=g).to(dt).to(dev)  # noqa: E731
    R = T * K2
    idx = torch.stack([torch.randperm(E, generator=g)[:K2] for _ in range(T)]).to(dev)
    se, ss, off, inv = torch.ops.zmoe.flatten_sort_count(idx, E)
    w = torch.rand(T, K2, generator=g).to(dev)
    rows = torch.randperm(T + 9, generator=g)[:T].to(dev)
    x, H, A, Y = r(T, d), r(R, 2 * f), r(R, f), r(R, d)
    W1, W2 = r(E, 2 * f, d), r(E, d, f)
    logits = r(T, E)
    p = torch.rand(T, K2, generator=g).to(dev)
    wide = r(T, d + 8)[:, :d]                 # rows 8 elements further apart than they are long
    ops = {
        "route_topk": (logits, r(E, dt=torch.float32), K2, dtype == torch.bfloat16),
        "route_topk_backward": (w, p, idx, E, x),
        "flatten_sort_count": (idx, E),
        "flatten_sort_count_weights": (idx, w, E),
        "grouped_mm": (A, W2.permute(0, 2, 1), se, ss, 1, True, False, off, "scatter2scatter"),
        "group_bwd_w": (Y, wide, off, E, ss, K2, False),
        "group_bwd_w_bias": (Y, x, off, E, ss, K2),
        "dense_wgrad": (r(3000, d), r(3000, f), False),
        "combine": (Y, w, K2, x, None, 0),
        "combine_rows": (Y, None, K2, None, rows, T + 9),
        "combine_backward": (Y, x, w, inv, None),
        "combine_backward_rows": (Y, r(T + 9, d), w, inv, rows),
        "sum_k": (Y, K2, x, False),
        "swiglu": (H,),
        "swiglu_backward": (A, H),
        "swiglu_backward_gates": (A, H, w.reshape(-1), ss),
        "rmsnorm_rows": (wide, r(d), 1e-6, None),
        "rmsnorm_rows_backward": (x, r(T + 9, d), rows, torch.rand(T, generator=g).to(dev), r(d)),
    }
    if d % 8 == 0 and f % 8 == 0:             # widths that the fused kernels take
        ops["glu_w1_forward"] = (wide, W1, se, ss, off, K2, None)
        ops["glu_w2_backward_dh"] = (Y, W2, H, se, off)
        ops["swiglu_route_backward"] = (r(T, f), r(T, 2 * f), w, p, idx, E)
    if dtype == torch.float32:
        ops["cast_bf16"] = (x,)
    elif d % 8 == 0 and f % 8 == 0:
        ops["glu_w1_forward_scaled"] = (x, W1, se, ss, off, K2, w.reshape(-1)[ss])
        xs, ws, fs = r(8, 128), [r(E, 128, 128), r(E, 128, 64)], 192   # streaming sizes: 8 tokens, 2 of 8 experts
        i8 = idx[:8].contiguous()
        _, s8, o8, _ = torch.ops.zmoe.flatten_sort_count(i8, E)
        ops["glu_shared_forward"] = (xs, *ws, s8, o8, K2, torch.rand(8 * K2, generator=g).to(dev), r(fs, 128),
                                     r(fs, 128), r(128, fs))
        ops["group_bwd_w_f32"] = (Y, x, off, E, ss, K2, True)
        ops["group_bwd_w_gather_dy"] = (x, ss, K2, A, off, E, True)
        ops["dense_wgrad_f32"] = (r(5000, d), r(5000, f), True)
        ops["sum_k_f32"] = (Y, K2, None, True)
    return ops


def _name(key):
    for end in ("_scaled", "_f32", "_rows"):
        if key.endswith(end) and key != "rmsnorm_rows":
            return key[:-len(end)]
    return key


def _same(a, b):
    a, b = ([a], [b]) if isinstance(a, torch.Tensor) else (a, b)
    assert len(a) == len(b)
    for u, v in zip(a, b):
        assert u.dtype == v.dtype and u.shape == v.shape and u.stride() == v.stride()
        assert torch.equal(u, v)


def _no_general_form(monkeypatch):
    """Every function that the general forms are made of fails."""
    from zmoe import ops as zops

    def gone(*args, **kwargs):
        raise AssertionError("the general form ran")

    for n, v in list(vars(zops).items()):
        if callable(v) and getattr(v, "__module__", None) == zops.__name__:
            monkeypatch.setattr(zops, n, gone)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,f", [(D, F), (D + 3, F + 1)])
def test_native_op_equals_general(hip_device, dtype, d, f, monkeypatch):
    from zmoe import library as zl

    for key, args in _ops(hip_device, dtype, d, f).items():
        native, general = getattr(zl, _name(key)), getattr(torch.ops.zmoe, _name(key))
        try:
            ref = general(*args)
        except ValueError:
            assert (d, f) != (D, F), key  # only widths without a padded form are refused
            with pytest.raises(ValueError), torch.no_grad():
                native(*args)
            continue
        with torch.no_grad(), monkeypatch.context() as m:
            _no_general_form(m)
            _same(native(*args), ref)


def test_native_op_conversions_and_refusals(hip_device):
    from zmoe import library as zl
    from zmoe import profiling

    ops = _ops(hip_device, torch.bfloat16, D, F)
    Y, w, k, x, _, _ = ops["combine"]
    idx = ops["flatten_sort_count"][0]
    with torch.no_grad():
        # int32 ids, bf16 gates, an fp32 addend, a transposed operand: converted as before
        _same(zl.flatten_sort_count(idx.int(), E), torch.ops.zmoe.flatten_sort_count(idx.int(), E))
        args = (Y, w.bfloat16(), k, x.float(), None, 0)
        _same(zl.combine(*args), torch.ops.zmoe.combine(*args))
        Yt = Y.t().contiguous().t()
        _same(zl.sum_k(Yt, k, None, False), torch.ops.zmoe.sum_k(Yt, k, None, False))
        profiling.enable("sum_k")  # timed launches run the general form
        try:
            zl.sum_k(Y, k, None, False)
            assert len(profiling.durations_ms("sum_k")) == 1
        finally:
            profiling.disable()
            profiling.reset()
        for bad in (lambda: zl.swiglu(Y.half()), lambda: zl.swiglu(Y.cpu()),
                    lambda: zl.route_topk(ops["route_topk"][0], ops["route_topk"][1][:-1], K2, True),
                    lambda: zl.group_bwd_w_gather_dy(x.float(), idx.view(-1), K2, Y.float(), idx[0], E, False)):
            with pytest.raises(ValueError):
                bad()
    leaf = Y.clone().requires_grad_(True)
    with pytest.raises(RuntimeError):   # no formula: refused, not silently dropped
        zl.sum_k(leaf, k, None, False).sum().backward()


def _off(t, by=1):
    """A copy of ``t`` that starts ``by`` elements into a buffer."""
    buf = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)
    view = buf[by:].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_native_op_operands_off_16_bytes(hip_device, dtype, monkeypatch):
    """Rows have to start on 16 bytes in both forms; per-row floats, a norm's weight and the router's
    logits need not, natively."""
    from zmoe import library as zl

    ops = _ops(hip_device, dtype, D, F)
    for key in ("swiglu", "swiglu_backward", "swiglu_backward_gates", "combine", "sum_k", "rmsnorm_rows",
                "glu_w1_forward", "grouped_mm", "group_bwd_w", "dense_wgrad", "cast_bf16"):
        if key in ops:
            args = (_off(ops[key][0]), *ops[key][1:])
            for form in (getattr(zl, key), getattr(torch.ops.zmoe, key)):
                with pytest.raises(ValueError), torch.no_grad():
                    form(*args)
    for key, at in (("route_topk", 0), ("combine", 1), ("swiglu_backward_gates", 2), ("flatten_sort_count_weights", 1),
                    ("rmsnorm_rows", 1), ("rmsnorm_rows_backward", 4), ("rmsnorm_rows_backward", 3)):
        args = ops[key]
        ref = getattr(torch.ops.zmoe, key)(*args)
        with torch.no_grad(), monkeypatch.context() as m:
            _no_general_form(m)
            _same(getattr(zl, key)(*args[:at], _off(args[at]), *args[at + 1:]), ref)


def test_native_ops_on_streams_and_threads(hip_device):
    """An op runs on the caller's current stream, after what is queued there, also from several
    threads at once."""
    from zmoe import library as zl

    cases = []
    for key, args in _ops(hip_device, torch.bfloat16, D, F).items():
        cases.append((key, getattr(zl, _name(key)), args, getattr(torch.ops.zmoe, _name(key))(*args)))
    torch.cuda.synchronize()
    failed = []

    def work():
        stream = torch.cuda.Stream()
        try:
            with torch.no_grad(), torch.cuda.stream(stream):
                for key, native, args, ref in cases:
                    # the floating operands arrive late, on this stream
                    late = [torch.zeros_like(a) if isinstance(a, torch.Tensor) and a.is_floating_point() else a
                            for a in args]
                    torch.cuda._sleep(2_000_000)
                    for a, b in zip(late, args):
                        if a is not b:
                            a.copy_(b)
                    got = native(*late)
                    stream.synchronize()
                    _same(got, ref)
        except Exception as e:  # reported by the main thread
            failed.append((key, e))

    work()
    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


def test_native_mutating_ops(hip_device):
    from scattermoe.kernels import ops as ko

    ops = _ops(hip_device, torch.bfloat16, D, F)
    A, W2t, se, ss, _, xg, yg, off, _ = ops["grouped_mm"]
    b = torch.randn(E, D, generator=gen(3)).bfloat16().to(hip_device)
    Y, w = ops["combine"][:2]
    x = ops["combine"][3]
    grouped = lambda: ko.scatter2scatter(A, W2t, se, ss, 1, b=b, x_grouped=xg, y_grouped=yg,  # noqa: E731
                                         expert_offsets=off)
    calls = (grouped, lambda: ko.scatter2scatter(A, W2t, se, ss, 1, x_grouped=xg, y_grouped=yg),
             lambda: ko.rowwise_sum_product(Y.view(T, K2, D), x), lambda: ko.group(x, ss, w.view(-1), K2),
             lambda: ko.group(x, ss, None, K2), lambda: ko.group_bwd_W(Y, A, off, E, has_bias=True)[0],
             lambda: ko.group_bwd_W(Y, A, off, E, has_bias=True)[1])
    for call in calls:
        with torch.no_grad():
            got = call()
        _same(got, call())   # grad mode on: the general form
    out = torch.empty(T * K2, D, dtype=torch.bfloat16, device=hip_device)
    before = out._version
    with torch.no_grad():
        ko.group(x, ss, None, K2, out=out)
    assert out._version > before
