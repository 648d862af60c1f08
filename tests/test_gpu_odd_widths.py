"""Feature widths that are not whole 16-byte chunks (K, N or d not a multiple of 8 bf16 or 4
fp32 elements), which the reference's masked kernels accept (scattermoe/kernels/ops.py:159-179,
:404-435, :504-519): the op wrappers run them through zero-padded copies, and the modules fall
back from the fused paths to the module composition. Checked against the oracle at the
north-star tolerances."""

import numpy as np
import pytest
import torch

import oracle as O
from helpers import TOL, assert_close, assert_close_fro, gen, np64, random_topk

pytestmark = pytest.mark.gpu

# (K, N): every residue of 8 appears in K or N; fp32 rows need multiples of 4
WIDTHS = [(100, 37), (13, 200), (257, 259), (6, 3), (130, 66), (41, 255), (7, 128), (64, 17)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N", WIDTHS)
@pytest.mark.parametrize("xg,yg", [(False, True), (True, False), (False, False)])
def test_scatter2scatter_any_width(hip_device, dtype, K, N, xg, yg):
    from zmoe import ops

    T, E, k = 300, 8, 2
    idx = random_topk(T, E, k, seed=K + N, skew=0.5)
    se, ss, off, _ = ops.flatten_sort_count(idx.to(hip_device), E)
    g = gen(K * 7 + N)
    X = torch.randn(T * k if xg else T, K, generator=g).to(dtype)
    Wp = (torch.randn(E, N, K, generator=g) / K ** 0.5).to(dtype)
    b = (torch.randn(E, N, generator=g) * 0.3).to(dtype)
    Y = ops.scatter2scatter(X.to(hip_device), Wp.to(hip_device).permute(0, 2, 1), se, ss, 1 if xg else k,
                            b=b.to(hip_device), x_grouped=xg, y_grouped=yg, expert_offsets=off)
    assert Y.shape == (T * k, N)
    ref = O.scatter2scatter(np64(X), np64(Wp).transpose(0, 2, 1), se.cpu().numpy(), ss.cpu().numpy(),
                            1 if xg else k, b=np64(b), x_grouped=xg, y_grouped=yg)
    assert_close(np64(Y), ref, **TOL[dtype], what=f"scatter2scatter K={K} N={N}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N", WIDTHS)
def test_group_bwd_w_any_width(hip_device, dtype, K, N):
    from zmoe import ops

    T, E, k = 300, 8, 3
    idx = random_topk(T, E, k, seed=3 * K + N, skew=1.0)
    se, ss, off, _ = ops.flatten_sort_count(idx.to(hip_device), E)
    g = gen(K + 11 * N)
    DY = torch.randn(T * k, N, generator=g).to(dtype)
    X = torch.randn(T, K, generator=g).to(dtype)
    DWt, Db = ops.group_bwd_w(DY.to(hip_device), X.to(hip_device), off, E, has_bias=True, x_gather=ss, x_div=k)
    assert DWt.shape == (E, N, K) and DWt.is_contiguous() and Db.shape == (E, N)
    ref, rb = O.group_bwd_w(np64(DY), O.group(np64(X), ss.cpu().numpy(), fan_out=k), off.cpu().numpy(), E,
                            has_bias=True)
    if dtype == torch.float32:
        assert_close_fro(np64(DWt), ref.transpose(0, 2, 1), what="group_bwd_w f32")
    else:
        assert_close(np64(DWt), ref.transpose(0, 2, 1), **TOL[dtype], what=f"group_bwd_w K={K} N={N}")
    assert_close(np64(Db), rb, **TOL[dtype], what="bias grad")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [3, 37, 100, 255])
def test_row_passes_any_width(hip_device, dtype, d):
    """group (with coefficients), combine (gates, addend, padded output rows) and the k-sum."""
    from zmoe import ops

    T, k = 211, 4
    g = gen(d)
    A = torch.randn(T, d, generator=g).to(dtype)
    perm = torch.randperm(T * k, generator=g)
    c = torch.rand(T * k, generator=g)
    Y = ops.group(A.to(hip_device), perm.to(hip_device), coeff=c.to(hip_device), fan_out=k)
    assert_close(np64(Y), O.group(np64(A), perm.numpy(), coeff=c.double().numpy(), fan_out=k), **TOL[dtype],
                 what="group")
    Ye = torch.randn(T * k, d, generator=g).to(dtype)
    gates = torch.rand(T, k, generator=g)
    add = torch.randn(T, d, generator=g).to(dtype)
    rows = torch.randperm(T + 50, generator=g)[:T]
    out = ops.combine(Ye.to(hip_device), gates.to(hip_device), k, add.to(hip_device), rows.to(hip_device), T + 50)
    ref = np.zeros((T + 50, d))
    ref[rows.numpy()] = np64(add) + np.einsum("tj,tjd->td", gates.double().numpy(), np64(Ye).reshape(T, k, d))
    assert_close(np64(out), ref, **TOL[dtype], what="combine")
    s = ops.sum_k(Ye.to(hip_device), k, add.to(hip_device))
    assert_close(np64(s), np64(Ye).reshape(T, k, d).sum(1) + np64(add), **TOL[dtype], what="sum_k")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_glumlp_odd_widths(hip_device, dtype):
    """GLUMLP(input_size=100, hidden_size=52): the fused path declines these widths and the
    module composition runs, forward and backward, against the oracle."""
    from scattermoe.mlp import GLUMLP

    torch.manual_seed(5)
    T, d, f, E, k = 400, 100, 52, 8, 2
    mlp = GLUMLP(d, f, E, k).to(hip_device).to(dtype)
    x = torch.randn(T, d, device=hip_device).to(dtype).requires_grad_(True)
    idx = random_topk(T, E, k, seed=9).to(hip_device)
    p = (torch.rand(T, k, generator=gen(4)) + 0.1).to(hip_device)
    y = mlp(x, p, idx)
    dy = torch.randn(T, d, generator=gen(6)).to(dtype).to(hip_device)
    y.backward(dy)
    bf16 = dtype == torch.bfloat16
    ry, cache = O.glu_mlp_forward(np64(x), p.double().cpu().numpy(), idx.cpu().numpy(), np64(mlp.experts.weight),
                                  np64(mlp.output_experts.weight), store="bf16" if bf16 else None)
    rdx, rdW1, rdW2, _, rss = O.glu_mlp_backward(np64(dy), cache, rss=True)
    tol = TOL[dtype]
    assert_close(np64(y), ry, **tol, what="y")
    assert_close(np64(x.grad), rdx, **tol, what="dx")
    if bf16:  # the composition rounds silu(gate) and the product as two bf16 ops: two rss allowances
        assert_close(np64(mlp.experts.weight.grad), rdW1, **tol, what="dW1", rss=2 * rss["W1"])
        assert_close(np64(mlp.output_experts.weight.grad), rdW2, **tol, what="dW2", rss=2 * rss["W2"])
    else:
        assert_close_fro(np64(mlp.experts.weight.grad), rdW1, what="dW1")
        assert_close_fro(np64(mlp.output_experts.weight.grad), rdW2, what="dW2")


def test_moe_layer_odd_hidden_size(hip_device):
    """MoELayer with hidden_size = 100 and intermediate_size = 36 (bf16), forward and backward:
    the whole-layer function declines these widths; the composition's routing is bit-exact
    and its output and grads are within the bf16 bound of the oracle."""
    from modeling.model_config import ModelConfig
    from modeling.moe_layer import MoELayer

    torch.manual_seed(8)
    d, f, E, k = 100, 36, 12, 3
    cfg = ModelConfig(hidden_size=d, intermediate_size=f, n_experts=E + 1, n_shared_experts=1,
                      n_experts_per_token=k)
    layer = MoELayer(cfg).to(hip_device).to(torch.bfloat16)
    layer.gate.expert_biases.data = (0.1 * torch.randn(E)).to(hip_device)
    T = 500
    x = torch.randn(1, T, d, device=hip_device).to(torch.bfloat16).requires_grad_(True)
    out, idx = layer(x)
    dout = torch.randn(1, T, d, device=hip_device).to(torch.bfloat16)
    out.backward(dout)
    se = layer.shared_experts
    with torch.no_grad():
        logits = torch.nn.functional.linear(x.detach().view(T, d), layer.gate.weight).float().cpu().numpy()
    orc = O.MoELayerOracle(np64(layer.gate.weight), layer.gate.expert_biases.cpu().numpy(),
                           np64(layer.routed_experts.experts.weight), np64(layer.routed_experts.output_experts.weight),
                           k, shared=(np64(se.gate_proj.weight), np64(se.up_proj.weight), np64(se.down_proj.weight)),
                           round_probs_bf16=True, store="bf16", gate_scale_on="Y")
    rout, ridx, _ = orc.forward(np64(x.view(T, d)), logits=logits)
    np.testing.assert_array_equal(idx.view(T, k).cpu().numpy(), ridx)
    tol = TOL[torch.bfloat16]
    assert_close(np64(out.view(T, d)), rout, **tol, what="out")
    g = orc.backward(np64(dout.view(T, d)), rss=True)
    assert_close(np64(x.grad.view(T, d)), g["x"], **tol, what="dx")
    keys = {"gate.weight": "gate_weight", "routed_experts.experts.weight": "W1",
            "routed_experts.output_experts.weight": "W2", "shared_experts.gate_proj.weight": "shared_gate",
            "shared_experts.up_proj.weight": "shared_up", "shared_experts.down_proj.weight": "shared_down"}
    for n, p in layer.named_parameters():
        # the composition rounds a few more intermediates than the oracle models (torch's silu
        # and product as separate bf16 ops): two rss allowances, as for the two-path comparison
        assert_close(np64(p.grad), g[keys[n]], **tol, what=n, rss=2 * g["rss"][keys[n]])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,rows,cols,drows,dcols", [
    (1, 5, 1, 5, 8), (1, 1, 1031, 1, 1032), (3, 7, 513, 9, 516), (2, 6, 40, 5, 33), (1, 4, 512, 4, 511),
    (1, 0, 9, 3, 9), (2, 3, 0, 3, 4), (1, 300001, 3, 300002, 8), (3, 100001, 5, 100000, 3)])
def test_copy_pad(hip_device, dtype, batch, rows, cols, drows, dcols):
    """The padded copy at its edges: one element, partial last chunks on either side, zero rows and
    columns, cuts, more rows than one launch takes; a source that is a view starting off a 16-byte
    boundary with rows further apart than they are long, into a NaN-filled output."""
    from zmoe import ops

    wide = torch.randn(batch, rows + 1, cols + 3, generator=gen(rows + cols)).to(dtype).to(hip_device)
    src = wide[:, 1:, 1:cols + 1]
    out = torch.full((batch, drows, dcols), float("nan"), dtype=dtype, device=hip_device)
    ops.copy_pad(src, drows, dcols, out)
    ref = torch.zeros(batch, drows, dcols, dtype=dtype, device=hip_device)
    r, c = min(rows, drows), min(cols, dcols)
    ref[:, :r, :c] = src[:, :r, :c]
    assert torch.equal(out, ref)


def test_copy_pad_is_one_launch(hip_device):
    """Any number of rows goes in one launch (also many small matrices: a captured graph's nodes)."""
    import ctypes

    from zmoe import _lib, ops

    src = torch.randn(300, 1001, 5, device=hip_device)
    out = torch.empty(300, 1002, 8, device=hip_device)       # 300600 rows, more than a grid's y takes by fours
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        ops.copy_pad(src, 1002, 8, out)
    nodes = ctypes.c_size_t(0)
    # (the library's handle resolves the runtime that it is linked to)
    rc = _lib.load().hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes))
    assert rc == 0 and nodes.value == 1
    graph.instantiate()
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[:, :1001, :5], src)
        assert not out[:, 1001:].any() and not out[:, :, 5:].any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N", [8, 32, 40, 64, 136])
def test_bias_grad_row_counts(hip_device, dtype, N):
    """The bias grad where its rows are split differently: no rows, one, around the 128 row slots
    of a block and the four rows a slot loads at once; column counts around a block's 128 bytes."""
    from zmoe import ops

    counts = [0, 1, 127, 128, 129, 0, 511, 513, 1300]
    off = torch.tensor(np.cumsum(counts), device=hip_device)
    g = gen(N)
    DY = torch.randn(sum(counts), N, generator=g).to(dtype)
    X = torch.randn(sum(counts), 16, generator=g).to(dtype)
    _, Db = ops.group_bwd_w(DY.to(hip_device), X.to(hip_device), off, len(counts), has_bias=True)
    ref = np.stack([r.sum(0) for r in np.split(np64(DY), np.cumsum(counts)[:-1])])
    # fp32 sums of up to 1300 terms ~ N(0, 1): 1300 * 2^-24 * sum|terms| bounds any order
    atol = max(TOL[dtype]["atol"], 1300 * 2.0 ** -24 * float(np.abs(np64(DY)).sum(0).max()))
    assert_close(np64(Db), ref, rtol=TOL[dtype]["rtol"], atol=atol, what="bias grad")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("counts,N", [([0, 1, 31, 32, 33, 0, 31], 264), ([0, 128], 8), ([3] * 40, 72),   # <= 128 rows
                                      ([0, 1, 31, 32, 33, 127, 129, 400] * 16, 1024 + 8),     # wide blocks
                                      ([257] + [0] * 255, 1024), ([1] * 129, 2000),
                                      ([0, 33, 1, 0] + [1] * 90, 2000)])                       # both
def test_bias_grad_block_shapes(hip_device, dtype, counts, N):
    """The bias grad's other blocks: 256 threads where no expert can have more than 128 rows, and 512
    bytes of columns where there are many; rows around a slot's four and a block's pass over them."""
    from zmoe import ops

    off = torch.tensor(np.cumsum(counts), device=hip_device)
    g = gen(N + len(counts))
    DY = torch.randn(sum(counts), N, generator=g).to(dtype)
    X = torch.randn(sum(counts), 16, generator=g).to(dtype)
    _, Db = ops.group_bwd_w(DY.to(hip_device), X.to(hip_device), off, len(counts), has_bias=True)
    ref = np.stack([r.sum(0) for r in np.split(np64(DY), np.cumsum(counts)[:-1])])
    # fp32 sums of n terms: n * 2^-24 * sum|terms| bounds any order
    atol = max(TOL[dtype]["atol"], max(counts) * 2.0 ** -24 * float(np.abs(np64(DY)).sum(0).max()))
    assert_close(np64(Db), ref, rtol=TOL[dtype]["rtol"], atol=atol, what="bias grad")
