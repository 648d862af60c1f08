"""The layer's HIP entry points as ``torch.library`` custom ops (namespace ``zmoe``).

The reference keeps its layer compile-friendly by registering its kernels as custom
ops with fake implementations (scattermoe/kernels/ops.py:21, :212, :274, :461;
scattermoe/parallel_experts.py:6, :17) and compiles the whole forward
(main.py:929). These are the functional (non-mutating) ops that the autograd
functions of ``modeling.moe_layer``, ``scattermoe.mlp`` and ``zmoe.functional``
call: ``torch.compile`` sees each launch as one opaque node whose output shapes come
from the fake implementation, so tracing the layer needs no graph break and no host
sync. Each op runs the ``zmoe.ops`` wrapper of the same name (the C ABI through
ctypes) on the current stream, or, in eager calls with gradients off that nothing watches,
its native form (``LayerOp``).
"""

from __future__ import annotations

import inspect
import os
import threading
from typing import List, Optional

import torch
from torch.utils._device import DeviceContext

from . import _lib as L
from . import ops as _z
from . import profiling

_I64 = torch.int64
_F32 = torch.float32

_eager_loaded = False
_eager_lock = threading.Lock()


def _load_eager():
    """The native ops (csrc/eager_ops.cpp), loaded once; there is no fallback if they are missing."""
    global _eager_loaded
    with _eager_lock:
        if not _eager_loaded:
            L.load()  # the C ABI library they call
            if not os.path.exists(L.EAGER_PATH):
                raise ImportError(f"{os.path.basename(L.EAGER_PATH)} not found at {L.EAGER_PATH}; build it first "
                                  "(python architecture-zarelga-superposition_amd/build_lib.py)")
            torch.ops.load_library(L.EAGER_PATH)
            _eager_loaded = True


# Argument types that a native op takes. Others go to the custom_op: fake tensors and other subclasses
# with a __torch_dispatch__ or __torch_function__ of their own, and symbolic sizes.
_plain = frozenset((torch.Tensor, torch.nn.Parameter, int, bool, float, str, list, tuple, type(None))).issuperset

_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
_tracing, _transforms = torch._C._is_tracing, torch._C._functorch.get_dynamic_layer_stack_depth
_compiling, _grad_enabled, _forward_ad = torch.compiler.is_compiling, torch.is_grad_enabled, torch.autograd.forward_ad


def _watched_by_function_mode() -> bool:
    """Whether a torch-function mode is active besides a default device's, which watches no op."""
    return any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(_function_modes()))


class LayerOp(torch.library.CustomOpDef):
    """The custom op ``zmoe::<name>``, whose eager calls with gradients off run the native
    ``zmoe_eager::<name>`` of csrc/eager_ops.cpp.

    The layer calls its ops from inside autograd functions, where grad mode is off and there is
    nothing to record; a small layer's step is bound by the host time of its ~25 calls, most of
    it custom_op's Python (autograd kernel, redispatch, alias check) and the wrapper's. With
    grad mode on (a caller outside an autograd function, or a backward with create_graph) the
    call goes to the custom_op, which refuses a backward through it. So does a call that is
    observed by what knows the ops by their zmoe:: names or has rules registered on them (a
    compiler or tracer, a dispatch or function mode, a functorch transform, forward-mode AD), and
    one that zmoe.profiling times."""

    def __call__(self, *args, **kwargs):
        if (_compiling() or _grad_enabled() or kwargs or _dispatch_modes() or _transforms()
                or _forward_ad._current_level >= 0 or _tracing() or profiling.active()
                or not _plain(map(type, args)) or (_function_modes() and _watched_by_function_mode())
                or (self._lists and not all(_plain(map(type, args[i])) for i in self._lists if i < len(args)))):
            return super().__call__(*args, **kwargs)
        if self._native is None:
            _load_eager()
            # (the dispatcher's call itself: the overload object's Python __call__ only forwards to it)
            self._native = getattr(torch.ops.zmoe_eager, self._name).default._op
        out = self._native(*args)
        for i in self._mutated:  # as custom_op does: autograd sees that the tensor changed
            if i < len(args) and args[i] is not None:
                torch.autograd.graph.increment_version(args[i])
        return out


def layer_op(name: str, mutates_args=()):
    """Decorator: ``torch.library.custom_op("zmoe::<name>")`` as a ``LayerOp``."""

    def wrap(fn):
        op = torch.library.custom_op(f"zmoe::{name}", mutates_args=mutates_args)(fn)
        op.__class__ = LayerOp
        op._native = None
        params = inspect.signature(fn).parameters
        op._mutated = tuple(i for i, p in enumerate(params) if p in mutates_args)
        op._lists = tuple(i for i, p in enumerate(params.values()) if str(p.annotation).startswith("List["))
        return op

    return wrap


def _empty(shape, like: torch.Tensor, dtype=None):
    return torch.empty(shape, dtype=dtype or like.dtype, device=like.device)


# ------------------------------------------------------------------ routing
@layer_op("route_topk")
def route_topk(logits: torch.Tensor, expert_biases: torch.Tensor, k: int,
               round_probs_bf16: bool) -> List[torch.Tensor]:
    """moe_gate.py:27-34 from the logits: [idx int64, weight f32, prob f32], each [T, k]."""
    return list(_z.route_topk(logits, expert_biases, k, round_probs_bf16=round_probs_bf16))


@route_topk.register_fake
def _(logits, expert_biases, k, round_probs_bf16):
    T = logits.shape[0]
    return [_empty((T, k), logits, _I64), _empty((T, k), logits, _F32), _empty((T, k), logits, _F32)]


@layer_op("swiglu_route_backward")
def swiglu_route_backward(dAs: torch.Tensor, Hs: torch.Tensor, d_gates: torch.Tensor, topk_prob: torch.Tensor,
                          topk_idx: torch.Tensor, num_experts: int) -> torch.Tensor:
    """[swiglu_backward(dAs, Hs) | d_logits] side by side in one [T, 2f + E] buffer: the
    shared expert's dH and the routing backward (autograd of moe_gate.py:27-34)."""
    T, two_f = Hs.shape
    G = torch.empty((T, two_f + num_experts), dtype=Hs.dtype, device=Hs.device)
    _z.swiglu_backward(dAs, Hs, out=G[:, :two_f])
    _z.route_topk_backward(d_gates, topk_prob, topk_idx, num_experts, Hs.dtype, out=G[:, two_f:])
    return G


@swiglu_route_backward.register_fake
def _(dAs, Hs, d_gates, topk_prob, topk_idx, num_experts):
    return _empty((Hs.shape[0], Hs.shape[1] + num_experts), Hs)


@layer_op("route_topk_backward")
def route_topk_backward(d_weight: torch.Tensor, topk_prob: torch.Tensor, topk_idx: torch.Tensor, num_experts: int,
                        like: torch.Tensor) -> torch.Tensor:
    """d_logits [T, E] in ``like``'s dtype."""
    return _z.route_topk_backward(d_weight, topk_prob, topk_idx, num_experts, like.dtype)


@route_topk_backward.register_fake
def _(d_weight, topk_prob, topk_idx, num_experts, like):
    return _empty((topk_idx.shape[0], num_experts), like)


# ------------------------------------------------------------------ sort
@layer_op("flatten_sort_count")
def flatten_sort_count(expert_idxs: torch.Tensor, num_experts: int) -> List[torch.Tensor]:
    """parallel_experts.py:21-28: [sorted_expert_idxs, sorted_scattered_idxs, expert_offsets,
    inverse int32]."""
    return list(_z.flatten_sort_count(expert_idxs, num_experts))


@flatten_sort_count.register_fake
def _(expert_idxs, num_experts):
    R = expert_idxs.numel()
    return [_empty((R,), expert_idxs, _I64), _empty((R,), expert_idxs, _I64),
            _empty((num_experts,), expert_idxs, _I64), _empty((R,), expert_idxs, torch.int32)]


@layer_op("flatten_sort_count_weights")
def flatten_sort_count_weights(expert_idxs: torch.Tensor, weights: torch.Tensor,
                               num_experts: int) -> List[torch.Tensor]:
    """flatten_sort_count's four, and the routing weights in sorted order."""
    return list(_z.flatten_sort_count_weights(expert_idxs, weights, num_experts))


@flatten_sort_count_weights.register_fake
def _(expert_idxs, weights, num_experts):
    R = expert_idxs.numel()
    return [_empty((R,), expert_idxs, _I64), _empty((R,), expert_idxs, _I64),
            _empty((num_experts,), expert_idxs, _I64), _empty((R,), expert_idxs, torch.int32),
            _empty((R,), expert_idxs, _F32)]


# ------------------------------------------------------------------ grouped GEMMs
glu_stream_shared_ok = _z.glu_stream_shared_ok
glu_stream_shared_pays = _z.glu_stream_shared_pays


@layer_op("glu_shared_forward")
def glu_shared_forward(x: torch.Tensor, W1: torch.Tensor, W2: torch.Tensor, sorted_scattered_idxs: torch.Tensor,
                       expert_offsets: torch.Tensor, k: int, row_scale: torch.Tensor, W_up: torch.Tensor,
                       W_gate: torch.Tensor, W_down: torch.Tensor) -> List[torch.Tensor]:
    """Few rows per expert: the routed and shared experts' forward in two launches:
    [H, A, Y (slot order), Hs, As, S]."""
    return list(_z.glu_shared_forward(x, W1, W2, sorted_scattered_idxs, expert_offsets, k, row_scale, W_up, W_gate,
                                      W_down))


@glu_shared_forward.register_fake
def _(x, W1, W2, sorted_scattered_idxs, expert_offsets, k, row_scale, W_up, W_gate, W_down):
    T, d = x.shape
    R, two_f, fs = T * k, W1.shape[1], W_up.shape[0]
    return [_empty((R, two_f), x), _empty((R, two_f // 2), x), _empty((R, d), x), _empty((T, 2 * fs), x),
            _empty((T, fs), x), _empty((T, d), x)]


@layer_op("glu_w1_forward")
def glu_w1_forward(x: torch.Tensor, W1: torch.Tensor, sorted_expert_idxs: torch.Tensor,
                   sorted_scattered_idxs: torch.Tensor, expert_offsets: torch.Tensor, k: int,
                   row_scale: Optional[torch.Tensor]) -> List[torch.Tensor]:
    """W1 grouped GEMM with the SwiGLU epilogue: [H [T*k, 2f], A [T*k, f]] (A scaled by
    ``row_scale`` when given)."""
    return list(_z.glu_w1_forward(x, W1, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, k,
                                  row_scale=row_scale))


@glu_w1_forward.register_fake
def _(x, W1, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, k, row_scale):
    R = x.shape[0] * k
    two_f = W1.shape[1]
    return [_empty((R, two_f), x), _empty((R, two_f // 2), x)]


@layer_op("glu_act_forward")
def glu_act_forward(x: torch.Tensor, W1: torch.Tensor, sorted_scattered_idxs: torch.Tensor,
                    expert_offsets: torch.Tensor, k: int, row_scale: Optional[torch.Tensor]) -> torch.Tensor:
    """``glu_w1_forward``'s A alone, for a forward whose backward will not run."""
    return _z.glu_act_forward(x, W1, sorted_scattered_idxs, expert_offsets, k, row_scale)


@glu_act_forward.register_fake
def _(x, W1, sorted_scattered_idxs, expert_offsets, k, row_scale):
    return _empty((x.shape[0] * k, W1.shape[1] // 2), x)


@layer_op("grouped_mm")
def grouped_mm(X: torch.Tensor, W: torch.Tensor, sorted_expert_idxs: torch.Tensor,
               sorted_scattered_idxs: torch.Tensor, k: int, x_grouped: bool, y_grouped: bool,
               expert_offsets: torch.Tensor, region: str) -> torch.Tensor:
    """scatter2scatter (ops.py:192-209) into a new [T*k, N] tensor; W the logical [E, K, N]."""
    return _z.scatter2scatter(X, W, sorted_expert_idxs, sorted_scattered_idxs, k, x_grouped=x_grouped,
                              y_grouped=y_grouped, expert_offsets=expert_offsets, region=region)


@grouped_mm.register_fake
def _(X, W, sorted_expert_idxs, sorted_scattered_idxs, k, x_grouped, y_grouped, expert_offsets, region):
    return _empty((sorted_expert_idxs.shape[0], W.shape[2]), X)


@layer_op("glu_w2_backward_dh")
def glu_w2_backward_dh(dYg: torch.Tensor, W2: torch.Tensor, H: torch.Tensor, sorted_expert_idxs: torch.Tensor,
                       expert_offsets: torch.Tensor) -> torch.Tensor:
    """dH [T*k, 2f]: the W2 input-grad GEMM with the SwiGLU backward epilogue."""
    return _z.glu_w2_backward_dh(dYg, W2, H, sorted_expert_idxs, expert_offsets)


@glu_w2_backward_dh.register_fake
def _(dYg, W2, H, sorted_expert_idxs, expert_offsets):
    return _empty(H.shape, dYg)


def _wdt(DY: torch.Tensor, out_f32: bool) -> torch.dtype:
    return torch.float32 if out_f32 else DY.dtype


@layer_op("group_bwd_w")
def group_bwd_w(DY: torch.Tensor, X: torch.Tensor, expert_offsets: torch.Tensor, num_experts: int,
                x_gather: Optional[torch.Tensor], x_div: int, out_f32: bool = False) -> torch.Tensor:
    """group_bwd_W (ops.py:263-271): DWt [E, N, K] (the parameter layout); ``out_f32``: fp32
    from the accumulators (bf16 operands, fp32 master weights)."""
    return _z.group_bwd_w(DY, X, expert_offsets, num_experts, x_gather=x_gather, x_div=x_div,
                          out_dtype=_wdt(DY, out_f32))[0]


@group_bwd_w.register_fake
def _(DY, X, expert_offsets, num_experts, x_gather, x_div, out_f32=False):
    return _empty((num_experts, DY.shape[1], X.shape[1]), DY, _wdt(DY, out_f32))


@layer_op("group_bwd_w_bias")
def group_bwd_w_bias(DY: torch.Tensor, X: torch.Tensor, expert_offsets: torch.Tensor, num_experts: int,
                     x_gather: Optional[torch.Tensor], x_div: int) -> List[torch.Tensor]:
    """group_bwd_W with has_bias (ops.py:263-271, :430-438): [DWt [E, N, K], Db [E, N]]."""
    return list(_z.group_bwd_w(DY, X, expert_offsets, num_experts, has_bias=True, x_gather=x_gather, x_div=x_div))


@group_bwd_w_bias.register_fake
def _(DY, X, expert_offsets, num_experts, x_gather, x_div):
    return [_empty((num_experts, DY.shape[1], X.shape[1]), DY), _empty((num_experts, DY.shape[1]), DY)]


@layer_op("group_bwd_w_gather_dy")
def group_bwd_w_gather_dy(DY: torch.Tensor, dy_gather: torch.Tensor, dy_div: int, X: torch.Tensor,
                          expert_offsets: torch.Tensor, num_experts: int, out_f32: bool = False) -> torch.Tensor:
    """Weight grads with DY's rows gathered in the kernel: DWt [E, N, K]."""
    return _z.group_bwd_w_gather_dy(DY, dy_gather, dy_div, X, expert_offsets, num_experts,
                                    out_dtype=_wdt(DY, out_f32))


@group_bwd_w_gather_dy.register_fake
def _(DY, dy_gather, dy_div, X, expert_offsets, num_experts, out_f32=False):
    return _empty((num_experts, DY.shape[1], X.shape[1]), DY, _wdt(DY, out_f32))


@layer_op("dense_wgrad")
def dense_wgrad(DY: torch.Tensor, X: torch.Tensor, out_f32: bool = False) -> torch.Tensor:
    """DW [N, K] = DY^T X (the F.linear weight grad, split-K)."""
    return _z.dense_wgrad(DY, X, out_dtype=_wdt(DY, out_f32))


@dense_wgrad.register_fake
def _(DY, X, out_f32=False):
    return _empty((DY.shape[1], X.shape[1]), DY, _wdt(DY, out_f32))


# ------------------------------------------------------------------ row passes
@layer_op("combine")
def combine(Y: torch.Tensor, gates: Optional[torch.Tensor], k: int, addend: Optional[torch.Tensor],
            out_rows: Optional[torch.Tensor], out_total: int) -> torch.Tensor:
    """out[t] = addend[t] + sum_j gates[t, j] Y[t*k + j] ([T, d], or the padded [out_total, d]
    when ``out_rows`` is given)."""
    return _z.combine(Y, gates, k, addend=addend, out_rows=out_rows, out_total=out_total if out_rows is not None
                      else None)


@combine.register_fake
def _(Y, gates, k, addend, out_rows, out_total):
    rows = out_total if out_rows is not None else Y.shape[0] // k
    return _empty((rows, Y.shape[1]), Y)


@layer_op("combine_backward")
def combine_backward(Y: torch.Tensor, grad_out: torch.Tensor, gates: torch.Tensor, inverse: torch.Tensor,
                     grad_rows: Optional[torch.Tensor]) -> List[torch.Tensor]:
    """[d_gates [T, k] f32, gate-scaled grad rows [T*k, d] in sorted order]."""
    return list(_z.combine_backward(Y, grad_out, gates, inverse, grad_rows=grad_rows))


@combine_backward.register_fake
def _(Y, grad_out, gates, inverse, grad_rows):
    T, k = gates.shape
    return [_empty((T, k), gates, _F32), _empty((T * k, Y.shape[-1]), Y)]


@layer_op("sum_k")
def sum_k(Xe: torch.Tensor, k: int, add0: Optional[torch.Tensor], out_f32: bool = False) -> torch.Tensor:
    """out[t] = sum_j Xe[t*k + j] (+ add0[t]) (parallel_experts.py:125); ``out_f32``: the fp32
    sum unrounded."""
    return _z.sum_k(Xe, k, add0=add0, out_dtype=torch.float32 if out_f32 else None)


@sum_k.register_fake
def _(Xe, k, add0, out_f32=False):
    return _empty((Xe.shape[0] // k, Xe.shape[1]), Xe, torch.float32 if out_f32 else None)


@layer_op("cast_bf16")
def cast_bf16(src: torch.Tensor) -> torch.Tensor:
    """The bf16 compute copy of an fp32 tensor (fp32 master weights under bf16 autocast)."""
    return _z.cast_bf16(src).clone() if src.dtype == torch.bfloat16 else _z.cast_bf16(src)


@cast_bf16.register_fake
def _(src):
    return _empty(src.shape, src, torch.bfloat16)


@layer_op("cast_bf16_packed")
def cast_bf16_packed(srcs: List[torch.Tensor], cat_from: int, any_from: int = -1) -> List[torch.Tensor]:
    """``cast_bf16`` of ``srcs[:cat_from]``, and of ``srcs[cat_from:]`` concatenated along dim 0;
    ``srcs[any_from:]`` (-1: the concatenated ones) may start at any element."""
    return list(_z.cast_bf16_packed(srcs, cat_from, any_from))


@cast_bf16_packed.register_fake
def _(srcs, cat_from, any_from=-1):
    tail = srcs[cat_from:]
    rows = sum(s.shape[0] for s in tail)
    return ([_empty(s.shape, s, torch.bfloat16) for s in srcs[:cat_from]]
            + [_empty((rows, *tail[0].shape[1:]), tail[0], torch.bfloat16)])


@layer_op("swiglu")
def swiglu(H: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up for H = [up | gate] (mlp.py:86, expert_layer.py:23-24)."""
    return _z.swiglu(H)


@swiglu.register_fake
def _(H):
    return _empty((H.shape[0], H.shape[1] // 2), H)


@layer_op("swiglu_backward")
def swiglu_backward(dA: torch.Tensor, H: torch.Tensor) -> torch.Tensor:
    return _z.swiglu_backward(dA, H)


@swiglu_backward.register_fake
def _(dA, H):
    return _empty(H.shape, H)


@layer_op("swiglu_backward_gates")
def swiglu_backward_gates(dA: torch.Tensor, H: torch.Tensor, row_scale: torch.Tensor,
                          slot_of_row: torch.Tensor) -> List[torch.Tensor]:
    """[dH [R, 2f], d_gates [R] f32 in slot order] of gate-scaled rows."""
    return list(_z.swiglu_backward_gates(dA, H, row_scale, slot_of_row))


@swiglu_backward_gates.register_fake
def _(dA, H, row_scale, slot_of_row):
    return [_empty(H.shape, H), _empty((H.shape[0],), H, _F32)]


@layer_op("rmsnorm_rows")
def rmsnorm_rows(X: torch.Tensor, weight: torch.Tensor, eps: float, rows: Optional[torch.Tensor]) -> List[torch.Tensor]:
    """[Y [n, d], rstd [n] f32]: zRMSNorm.py:10-17 on rows ``rows`` of X."""
    return list(_z.rmsnorm_rows(X, weight, eps, rows))


@rmsnorm_rows.register_fake
def _(X, weight, eps, rows):
    n = X.shape[0] if rows is None else rows.numel()
    return [_empty((n, X.shape[1]), X), _empty((n,), X, _F32)]


@layer_op("rmsnorm_rows_backward")
def rmsnorm_rows_backward(dY: torch.Tensor, X: torch.Tensor, rows: Optional[torch.Tensor], rstd: torch.Tensor,
                          weight: torch.Tensor) -> List[torch.Tensor]:
    """[dX [N, d] (zeros outside ``rows``), dweight]."""
    return list(_z.rmsnorm_rows_backward(dY, X, rows, rstd, weight))


@rmsnorm_rows_backward.register_fake
def _(dY, X, rows, rstd, weight):
    return [_empty(X.shape, X), _empty(weight.shape, weight)]
