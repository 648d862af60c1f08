// The layer's device ops as C++ dispatcher kernels (namespace zmoe_eager): what eager calls of
// zmoe/library.py run with gradients off, where no mode, tracer or transform watches. Each takes the
// operands that the layer itself passes (device tensors of one device, bf16 or f32 rows, int64 indices),
// allocates its outputs with torch and makes one C-ABI call on torch's current stream. Everything else
// (other dtypes and devices, strides the kernels do not take, bad sizes) goes to the op's general form,
// the Python wrapper registered as zmoe::<name>, which converts, pads or raises.
//
// Why native: a training step of a small layer is bound by its host work. An op costs ~20-40 us
// through torch.library.custom_op, the Python wrapper and ctypes, ~8 us here (the training step at
// d = 512, f = 160, 32 experts, 6.5 k tokens: 1013 -> 744 us of host time, a 4-token forward at
// d = 2048: 284 -> 179 us).
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <algorithm>
#include <limits>
#include <optional>
#include <string>
#include <vector>

#include "zmoe.h"

namespace {

using at::Tensor;
using Opt = std::optional<Tensor>;
using Tensors = std::vector<Tensor>;

// The op's general form, looked up once per call site.
template <typename Sig>
const c10::TypedOperatorHandle<Sig> general(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? ZMOE_DTYPE_BF16 : ZMOE_DTYPE_F32; }
int code(at::ScalarType t) { return t == at::kBFloat16 ? ZMOE_DTYPE_BF16 : ZMOE_DTYPE_F32; }
bool known(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat; }

bool fits_int(int64_t v) { return v >= std::numeric_limits<int>::min() && v <= std::numeric_limits<int>::max(); }

// A device tensor of `like`'s device.
bool on(const Tensor& t, const Tensor& like) { return t.is_cuda() && t.device() == like.device(); }
// Contiguous, of the given type, on `like`'s device.
bool flat(const Tensor& t, const Tensor& like, at::ScalarType dt) {
  return on(t, like) && t.scalar_type() == dt && t.is_contiguous();
}
// [rows, cols] with unit column stride, of like's dtype and device.
bool rows2(const Tensor& t, const Tensor& like) {
  return on(t, like) && t.scalar_type() == like.scalar_type() && t.dim() == 2 && t.stride(1) == 1;
}
bool index(const Tensor& t, const Tensor& like, int64_t n) { return flat(t, like, at::kLong) && t.numel() == n; }

Tensor empty(at::IntArrayRef shape, const Tensor& like, at::ScalarType dt) {
  return at::empty(shape, like.options().dtype(dt));
}
Tensor empty(at::IntArrayRef shape, const Tensor& like) { return at::empty(shape, like.options()); }
Tensor workspace(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)(bytes > 16 ? bytes : 16)}, like.options().dtype(at::kByte));
}

template <typename T> T* ptr(const Tensor& t) { return static_cast<T*>(t.data_ptr()); }
void* raw(const Tensor& t) { return t.data_ptr(); }
const int64_t* ids(const Tensor& t) { return ptr<const int64_t>(t); }

// ------------------------------------------------------------------ padded copies
// Widths that are not whole 16-byte chunks go through zero-padded copies, as in zmoe.ops.
int64_t vec(const Tensor& t) { return 16 / (int64_t)t.element_size(); }
int64_t up(int64_t n, const Tensor& like) { return (n + vec(like) - 1) / vec(like) * vec(like); }

// src [r, c] or [b, r, c] (unit last stride) -> dst [rows, cols] or [b, rows, cols], cut or
// zero-filled; false on an error.
bool copy_pad_into(const Tensor& src, const Tensor& dst) {
  const int64_t nd = src.dim();
  const int64_t rows = dst.size(-2), cols = dst.size(-1);
  return zmoe_copy_pad(raw(src), nd == 3 ? src.stride(0) : 0, src.stride(-2), nd == 3 ? src.size(0) : 1,
                       std::min(rows, src.size(-2)), std::min(cols, src.size(-1)), code(src), raw(dst), rows, cols,
                       stream_of(src)) == ZMOE_OK;
}
// The padded copy, or src itself where it has that size (undefined on an error).
Tensor padded(const Tensor& src, int64_t rows, int64_t cols) {
  if (src.size(-2) == rows && src.size(-1) == cols) return src;
  Tensor dst = src.dim() == 3 ? empty({src.size(0), rows, cols}, src) : empty({rows, cols}, src);
  return copy_pad_into(src, dst) ? dst : Tensor();
}

// ------------------------------------------------------------------ routing and sort
Tensors route_topk(const Tensor& logits, const Tensor& bias, int64_t k, bool round) {
  if (logits.is_cuda() && known(logits) && logits.dim() == 2 && logits.is_contiguous() &&
      flat(bias, logits, at::kFloat) && bias.numel() == logits.size(1) && k >= 0 && fits_int(k) &&
      fits_int(logits.size(1))) {
    const c10::DeviceGuard guard(logits.device());
    const int64_t T = logits.size(0);
    Tensor idx = empty({T, k}, logits, at::kLong), w = empty({T, k}, logits, at::kFloat),
           p = empty({T, k}, logits, at::kFloat);
    if (zmoe_route_topk(raw(logits), code(logits), T, (int)logits.size(1), (int)k, ptr<const float>(bias), round,
                        ptr<int64_t>(idx), ptr<float>(w), ptr<float>(p), stream_of(logits)) == ZMOE_OK)
      return {idx, w, p};
  }
  static const auto op = general<Tensors(const Tensor&, const Tensor&, c10::SymInt, bool)>("zmoe::route_topk");
  return op.call(logits, bias, k, round);
}

// d_logits into out [T, E] (rows `ld` elements apart); false where the general form has to run.
bool route_backward_into(const Tensor& dw, const Tensor& p, const Tensor& idx, int64_t E, void* out, int64_t ld,
                         at::ScalarType dt) {
  if (idx.dim() != 2 || !idx.is_cuda() || !idx.is_contiguous() || idx.scalar_type() != at::kLong ||
      !flat(dw, idx, at::kFloat) || !flat(p, idx, at::kFloat) || dw.numel() != idx.numel() ||
      p.numel() != idx.numel() || !fits_int(E) || !fits_int(idx.size(1)))
    return false;
  return zmoe_route_topk_backward(ptr<const float>(dw), ptr<const float>(p), ids(idx), idx.size(0), (int)E,
                                  (int)idx.size(1), out, ld, code(dt), stream_of(idx)) == ZMOE_OK;
}

Tensor route_topk_backward(const Tensor& dw, const Tensor& p, const Tensor& idx, int64_t E, const Tensor& like) {
  if (known(like) && idx.is_cuda() && idx.dim() == 2 && on(like, idx) && E >= 0) {
    const c10::DeviceGuard guard(idx.device());
    Tensor out = empty({idx.size(0), E}, like);
    if (route_backward_into(dw, p, idx, E, raw(out), E, like.scalar_type())) return out;
  }
  static const auto op =
      general<Tensor(const Tensor&, const Tensor&, const Tensor&, c10::SymInt, const Tensor&)>("zmoe::route_topk_backward");
  return op.call(dw, p, idx, E, like);
}

Tensor swiglu_route_backward(const Tensor& dAs, const Tensor& Hs, const Tensor& dg, const Tensor& p, const Tensor& idx,
                             int64_t E) {
  if (Hs.is_cuda() && known(Hs) && Hs.dim() == 2 && Hs.is_contiguous() && flat(dAs, Hs, Hs.scalar_type()) &&
      dAs.numel() * 2 == Hs.numel() && on(idx, Hs) && idx.dim() == 2 && idx.size(0) == Hs.size(0) && E >= 0) {
    const c10::DeviceGuard guard(Hs.device());
    const int64_t T = Hs.size(0), two_f = Hs.size(1), ld = two_f + E;
    Tensor G = empty({T, ld}, Hs);
    char* tail = static_cast<char*>(raw(G)) + two_f * G.element_size();
    if (zmoe_swiglu_backward(raw(dAs), raw(Hs), T, two_f / 2, code(Hs), raw(G), ld, stream_of(Hs)) == ZMOE_OK &&
        route_backward_into(dg, p, idx, E, tail, ld, Hs.scalar_type()))
      return G;
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                        c10::SymInt)>("zmoe::swiglu_route_backward");
  return op.call(dAs, Hs, dg, p, idx, E);
}

Tensors flatten_sort_count(const Tensor& e, int64_t E) {
  if (e.is_cuda() && e.scalar_type() == at::kLong && e.is_contiguous() && E >= 0 && fits_int(E)) {
    const c10::DeviceGuard guard(e.device());
    const int64_t R = e.numel();
    const size_t bytes = zmoe_sort_workspace_bytes(R, (int)E);
    Tensor se = empty({R}, e), ss = empty({R}, e), off = empty({E}, e), inv = empty({R}, e, at::kInt),
           ws = workspace(bytes, e);
    if (zmoe_flatten_sort_count(ids(e), R, (int)E, ptr<int64_t>(se), ptr<int64_t>(ss), ptr<int64_t>(off),
                                ptr<int32_t>(inv), raw(ws), bytes, stream_of(e)) == ZMOE_OK)
      return {se, ss, off, inv};
  }
  static const auto op = general<Tensors(const Tensor&, c10::SymInt)>("zmoe::flatten_sort_count");
  return op.call(e, E);
}

Tensors flatten_sort_count_weights(const Tensor& e, const Tensor& w, int64_t E) {
  if (e.is_cuda() && e.scalar_type() == at::kLong && e.is_contiguous() && E >= 0 && fits_int(E) &&
      flat(w, e, at::kFloat) && w.numel() == e.numel()) {
    const c10::DeviceGuard guard(e.device());
    const int64_t R = e.numel();
    const size_t bytes = zmoe_sort_workspace_bytes(R, (int)E);
    Tensor se = empty({R}, e), ss = empty({R}, e), off = empty({E}, e), inv = empty({R}, e, at::kInt),
           sw = empty({R}, e, at::kFloat), ws = workspace(bytes, e);
    if (zmoe_flatten_sort_count_weights(ids(e), ptr<const float>(w), R, (int)E, ptr<int64_t>(se), ptr<int64_t>(ss),
                                        ptr<int64_t>(off), ptr<int32_t>(inv), ptr<float>(sw), raw(ws), bytes,
                                        stream_of(e)) == ZMOE_OK)
      return {se, ss, off, inv, sw};
  }
  static const auto op = general<Tensors(const Tensor&, const Tensor&, c10::SymInt)>("zmoe::flatten_sort_count_weights");
  return op.call(e, w, E);
}

// ------------------------------------------------------------------ grouped GEMMs
Tensors glu_shared_forward(const Tensor& x, const Tensor& W1, const Tensor& W2, const Tensor& ss, const Tensor& off,
                           int64_t k, const Tensor& scale, const Tensor& Wu, const Tensor& Wg, const Tensor& Wd) {
  const auto bf = at::kBFloat16;
  if (x.is_cuda() && x.dim() == 2 && flat(x, x, bf) && flat(W1, x, bf) && flat(W2, x, bf) && flat(Wu, x, bf) &&
      flat(Wg, x, bf) && flat(Wd, x, bf) && W1.dim() == 3 && W2.dim() == 3 && Wu.dim() == 2 && Wg.dim() == 2 &&
      Wd.dim() == 2 && k > 0 && fits_int(k) && W1.size(1) % 2 == 0 && fits_int(W1.size(0))) {
    const int64_t T = x.size(0), d = x.size(1), E = W1.size(0), f = W1.size(1) / 2, fs = Wu.size(0), R = T * k;
    if (W1.size(2) == d && W2.size(0) == E && W2.size(1) == d && W2.size(2) == f && Wu.size(1) == d &&
        Wg.size(0) == fs && Wg.size(1) == d && Wd.size(0) == d && Wd.size(1) == fs && index(ss, x, R) &&
        index(off, x, E) && flat(scale, x, at::kFloat) && scale.numel() == R &&
        zmoe_glu_stream_shared_ok(T, d, f, fs, (int)E, (int)k)) {
      const c10::DeviceGuard guard(x.device());
      Tensor H = empty({R, 2 * f}, x), A = empty({R, f}, x), Y = empty({R, d}, x), Hs = empty({T, 2 * fs}, x),
             As = empty({T, fs}, x), S = empty({T, d}, x);
      if (zmoe_glu_w1_forward_shared(raw(x), raw(W1), ids(ss), ids(off), T, d, f, (int)E, (int)k,
                                     ptr<const float>(scale), raw(H), raw(A), raw(Wu), raw(Wg), fs, raw(Hs), raw(As),
                                     stream_of(x)) == ZMOE_OK &&
          zmoe_glu_w2_forward_shared(raw(A), raw(W2), ids(ss), ids(off), T, d, f, (int)E, (int)k, raw(Y), raw(As),
                                     raw(Wd), fs, raw(S), stream_of(x)) == ZMOE_OK)
        return {H, A, Y, Hs, As, S};
    }
  }
  static const auto op =
      general<Tensors(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, c10::SymInt,
                      const Tensor&, const Tensor&, const Tensor&, const Tensor&)>("zmoe::glu_shared_forward");
  return op.call(x, W1, W2, ss, off, k, scale, Wu, Wg, Wd);
}

Tensors glu_w1_forward(const Tensor& x, const Tensor& W1, const Tensor& se, const Tensor& ss, const Tensor& off,
                       int64_t k, const Opt& scale) {
  if (x.is_cuda() && known(x) && rows2(x, x) && flat(W1, x, x.scalar_type()) && W1.dim() == 3 && k > 0 && fits_int(k) &&
      W1.size(2) == x.size(1) && W1.size(1) % 2 == 0 && fits_int(W1.size(0))) {
    const int64_t T = x.size(0), E = W1.size(0), two_f = W1.size(1), d = W1.size(2), R = T * k;
    if (index(se, x, R) && index(ss, x, R) && index(off, x, E) &&
        (!scale || (flat(*scale, x, at::kFloat) && scale->numel() == R))) {
      const c10::DeviceGuard guard(x.device());
      Tensor H = empty({R, two_f}, x), A = empty({R, two_f / 2}, x);
      const int rc =
          scale ? zmoe_glu_w1_forward_scaled(raw(x), x.stride(0), raw(W1), ids(se), ids(ss), ids(off), T, d, two_f / 2,
                                             (int)E, (int)k, code(x), ptr<const float>(*scale), raw(H), raw(A),
                                             stream_of(x))
                : zmoe_glu_w1_forward(raw(x), x.stride(0), raw(W1), ids(se), ids(ss), ids(off), T, d, two_f / 2, (int)E,
                                      (int)k, code(x), raw(H), raw(A), stream_of(x));
      if (rc == ZMOE_OK) return {H, A};
    }
  }
  static const auto op = general<Tensors(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                         c10::SymInt, const Opt&)>("zmoe::glu_w1_forward");
  return op.call(x, W1, se, ss, off, k, scale);
}

Tensor glu_act_forward(const Tensor& x, const Tensor& W1, const Tensor& ss, const Tensor& off, int64_t k,
                       const Opt& scale) {
  if (x.is_cuda() && known(x) && rows2(x, x) && flat(W1, x, x.scalar_type()) && W1.dim() == 3 && k > 0 && fits_int(k) &&
      W1.size(2) == x.size(1) && W1.size(1) % 2 == 0 && fits_int(W1.size(0))) {
    const int64_t T = x.size(0), E = W1.size(0), f = W1.size(1) / 2, R = T * k;
    if (index(ss, x, R) && index(off, x, E) && (!scale || (flat(*scale, x, at::kFloat) && scale->numel() == R))) {
      const c10::DeviceGuard guard(x.device());
      Tensor A = empty({R, f}, x);
      if (zmoe_glu_act_forward(raw(x), x.stride(0), raw(W1), ids(ss), ids(off), T, x.size(1), f, (int)E, (int)k,
                               code(x), scale ? ptr<const float>(*scale) : nullptr, raw(A), stream_of(x)) == ZMOE_OK)
        return A;
    }
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, c10::SymInt,
                                        const Opt&)>("zmoe::glu_act_forward");
  return op.call(x, W1, ss, off, k, scale);
}

// out [R, N] = the grouped product; false where the general form has to run.
bool grouped_into(const Tensor& X, const Tensor& W, const Opt& b, const Tensor& se, const Tensor& ss, int64_t k,
                  bool xg, bool yg, const Tensor& off, const Tensor& out) {
  if (!(X.is_cuda() && known(X) && rows2(X, X) && on(W, X) && W.dim() == 3 && W.scalar_type() == X.scalar_type() &&
        (W.stride(1) == 1 || W.stride(2) == 1) && k > 0 && fits_int(k) && W.size(1) == X.size(1) &&
        fits_int(W.size(0)) && rows2(out, X)))
    return false;
  const int64_t M = X.size(0), E = W.size(0), K = W.size(1), N = W.size(2), R = M * k;
  if (!(index(se, X, R) && index(ss, X, R) && index(off, X, E) && out.size(0) == R && out.size(1) == N)) return false;
  if (b && !(flat(*b, X, X.scalar_type()) && b->dim() == 2 && b->size(0) == E && b->size(1) == N)) return false;
  const int64_t Kp = up(K, X), Np = up(N, X);
  if (Kp != K || Np != N) {
    if (!out.is_contiguous()) return false;
    const Tensor Xp = padded(X, M, Kp);
    // in its storage order: unit stride along K (the nn.Linear layout) or along N
    Tensor Wp = W.stride(1) == 1 ? padded(W.permute({0, 2, 1}), Np, Kp) : padded(W, Kp, Np);
    const Tensor bp = b ? padded(*b, E, Np) : Tensor();
    if (!Xp.defined() || !Wp.defined() || (b && !bp.defined())) return false;
    if (W.stride(1) == 1) Wp = Wp.permute({0, 2, 1});
    const Tensor Y = Np == N ? out : empty({R, Np}, X);
    return grouped_into(Xp, Wp, b ? Opt(bp) : std::nullopt, se, ss, k, xg, yg, off, Y) &&
           (Np == N || copy_pad_into(Y, out));
  }
  return zmoe_scatter2scatter(raw(X), X.stride(0), raw(W), W.stride(0), W.stride(1), W.stride(2), b ? raw(*b) : nullptr,
                              b ? b->stride(0) : 0, ids(se), ids(ss), ids(off), M, K, N, (int)E, (int)k, xg, yg,
                              code(X), raw(out), out.stride(0), stream_of(X)) == ZMOE_OK;
}

Tensor grouped_mm(const Tensor& X, const Tensor& W, const Tensor& se, const Tensor& ss, int64_t k, bool xg, bool yg,
                  const Tensor& off, c10::string_view region) {
  if (X.is_cuda() && X.dim() == 2 && W.dim() == 3) {
    const c10::DeviceGuard guard(X.device());
    Tensor out = empty({se.numel(), W.size(2)}, X);
    if (grouped_into(X, W, std::nullopt, se, ss, k, xg, yg, off, out)) return out;
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, c10::SymInt, bool,
                                        bool, const Tensor&, c10::string_view)>("zmoe::grouped_mm");
  return op.call(X, W, se, ss, k, xg, yg, off, region);
}

void scatter2scatter(const Tensor& out, const Tensor& W, const Tensor& X, int64_t k, const Tensor& se, const Tensor& ss,
                     const Opt& b, bool xg, bool yg, const Opt& off) {
  if (off && X.is_cuda()) {
    const c10::DeviceGuard guard(X.device());
    if (grouped_into(X, W, b, se, ss, k, xg, yg, *off, out)) return;
  }
  static const auto op =
      general<void(const Tensor&, const Tensor&, const Tensor&, c10::SymInt, const Tensor&, const Tensor&, const Opt&,
                   bool, bool, const Opt&)>("zmoe::scatter2scatter");
  op.call(out, W, X, k, se, ss, b, xg, yg, off);
}

Tensor glu_w2_backward_dh(const Tensor& dY, const Tensor& W2, const Tensor& H, const Tensor& se, const Tensor& off) {
  if (dY.is_cuda() && known(dY) && dY.dim() == 2 && dY.is_contiguous() && flat(W2, dY, dY.scalar_type()) &&
      W2.dim() == 3 && W2.size(1) == dY.size(1) && flat(H, dY, dY.scalar_type()) && H.dim() == 2 &&
      H.size(0) == dY.size(0) && H.size(1) == 2 * W2.size(2) && index(se, dY, dY.size(0)) &&
      index(off, dY, W2.size(0)) && fits_int(W2.size(0))) {
    const c10::DeviceGuard guard(dY.device());
    Tensor dH = empty(H.sizes(), dY);
    if (zmoe_glu_w2_backward_dh(raw(dY), raw(W2), raw(H), ids(se), ids(off), dY.size(0), W2.size(1), W2.size(2),
                                (int)W2.size(0), code(dY), raw(dH), stream_of(dY)) == ZMOE_OK)
      return dH;
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&)>(
      "zmoe::glu_w2_backward_dh");
  return op.call(dY, W2, H, se, off);
}

// dW [E, N, K] (and the bias grad [E, N] when given); false where the general form has to run.
bool wgrad_into(const Tensor& DY, const Tensor& X, const Tensor& off, int64_t E, const Opt& gather, int64_t div,
                const Tensor& dW, const Opt& db) {
  if (!(DY.is_cuda() && known(DY) && rows2(DY, DY) && rows2(X, DY) && index(off, DY, E) && fits_int(E) &&
        fits_int(div) && (gather ? index(*gather, DY, DY.size(0)) : X.size(0) == DY.size(0))))
    return false;
  const int64_t N = DY.size(1), K = X.size(1), Np = up(N, DY), Kp = up(K, X);
  if (Np != N || Kp != K) {
    const Tensor DYp = padded(DY, DY.size(0), Np), Xp = padded(X, X.size(0), Kp);
    if (!DYp.defined() || !Xp.defined()) return false;
    const Tensor dWp = empty({E, Np, Kp}, dW), dbp = db && Np != N ? empty({E, Np}, *db) : Tensor();
    return wgrad_into(DYp, Xp, off, E, gather, div, dWp, dbp.defined() ? Opt(dbp) : db) && copy_pad_into(dWp, dW) &&
           (!dbp.defined() || copy_pad_into(dbp, *db));
  }
  return zmoe_group_bwd_w(raw(DY), DY.stride(0), raw(X), X.stride(0), gather ? ids(*gather) : nullptr, (int)div,
                          ids(off), DY.size(0), DY.size(1), X.size(1), (int)E, code(DY), code(dW), raw(dW),
                          db ? raw(*db) : nullptr, stream_of(DY)) == ZMOE_OK;
}

// The weight grad's dtype: f32 asked of bf16 operands, else the operands'.
at::ScalarType wgrad_dtype(const Tensor& DY, bool out_f32) { return out_f32 ? at::kFloat : DY.scalar_type(); }

Tensor group_bwd_w(const Tensor& DY, const Tensor& X, const Tensor& off, int64_t E, const Opt& gather, int64_t div,
                   bool out_f32) {
  if (DY.is_cuda() && DY.dim() == 2 && X.dim() == 2 && E >= 0) {
    const c10::DeviceGuard guard(DY.device());
    Tensor dW = empty({E, DY.size(1), X.size(1)}, DY, wgrad_dtype(DY, out_f32));
    if (wgrad_into(DY, X, off, E, gather, div, dW, std::nullopt)) return dW;
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&, const Tensor&, c10::SymInt, const Opt&,
                                        c10::SymInt, bool)>("zmoe::group_bwd_w");
  return op.call(DY, X, off, E, gather, div, out_f32);
}

Tensors group_bwd_w_bias(const Tensor& DY, const Tensor& X, const Tensor& off, int64_t E, const Opt& gather,
                         int64_t div) {
  if (DY.is_cuda() && DY.dim() == 2 && X.dim() == 2 && E >= 0) {
    const c10::DeviceGuard guard(DY.device());
    Tensor dW = empty({E, DY.size(1), X.size(1)}, DY), db = empty({E, DY.size(1)}, DY);
    if (wgrad_into(DY, X, off, E, gather, div, dW, db)) return {dW, db};
  }
  static const auto op = general<Tensors(const Tensor&, const Tensor&, const Tensor&, c10::SymInt, const Opt&,
                                         c10::SymInt)>("zmoe::group_bwd_w_bias");
  return op.call(DY, X, off, E, gather, div);
}

Tensor group_bwd_w_gather_dy(const Tensor& DY, const Tensor& gather, int64_t div, const Tensor& X, const Tensor& off,
                             int64_t E, bool out_f32) {
  if (DY.is_cuda() && DY.scalar_type() == at::kBFloat16 && rows2(DY, DY) && rows2(X, DY) &&
      index(gather, DY, X.size(0)) && div > 0 && fits_int(div) && DY.size(0) * div >= X.size(0) && index(off, DY, E) &&
      fits_int(E)) {
    const c10::DeviceGuard guard(DY.device());
    Tensor dW = empty({E, DY.size(1), X.size(1)}, DY, wgrad_dtype(DY, out_f32));
    if (zmoe_group_bwd_w_gather_dy(raw(DY), DY.stride(0), ids(gather), (int)div, raw(X), X.stride(0), ids(off),
                                   X.size(0), DY.size(1), X.size(1), (int)E, code(DY), code(dW), raw(dW),
                                   stream_of(DY)) == ZMOE_OK)
      return dW;
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&, c10::SymInt, const Tensor&, const Tensor&,
                                        c10::SymInt, bool)>("zmoe::group_bwd_w_gather_dy");
  return op.call(DY, gather, div, X, off, E, out_f32);
}

Tensor dense_wgrad(const Tensor& DY, const Tensor& X, bool out_f32) {
  if (DY.is_cuda() && known(DY) && rows2(DY, DY) && rows2(X, DY) && X.size(0) == DY.size(0)) {
    const c10::DeviceGuard guard(DY.device());
    const int64_t M = DY.size(0), N = DY.size(1), K = X.size(1);
    int splits = 0;
    if (zmoe_dense_wgrad_splits(M, N, K, 256, &splits) == ZMOE_OK) {
      Tensor dW = empty({N, K}, DY, wgrad_dtype(DY, out_f32));
      const size_t bytes = zmoe_dense_wgrad_workspace_bytes(N, K, DY.scalar_type() == at::kBFloat16 ? splits : 0);
      Tensor ws = workspace(bytes, DY);
      if (zmoe_dense_wgrad(raw(DY), DY.stride(0), raw(X), X.stride(0), M, N, K, code(DY), code(dW), splits, raw(dW),
                           raw(ws), bytes, stream_of(DY)) == ZMOE_OK)
        return dW;
    }
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&, bool)>("zmoe::dense_wgrad");
  return op.call(DY, X, out_f32);
}

// ------------------------------------------------------------------ row passes
Tensor combine(const Tensor& Y, const Opt& gates, int64_t k, const Opt& addend, const Opt& out_rows,
               int64_t out_total) {
  if (Y.is_cuda() && known(Y) && Y.dim() == 2 && Y.is_contiguous() && k > 0 && fits_int(k) && Y.size(0) % k == 0) {
    const int64_t T = Y.size(0) / k, d = Y.size(1);
    if ((!gates || (flat(*gates, Y, at::kFloat) && gates->numel() == T * k)) &&
        (!addend || (flat(*addend, Y, Y.scalar_type()) && addend->numel() == T * d)) &&
        (!out_rows || (index(*out_rows, Y, T) && out_total >= 0))) {
      const c10::DeviceGuard guard(Y.device());
      if (const int64_t dp = up(d, Y); dp != d) {
        const Tensor Yp = padded(Y, T * k, dp);
        const Tensor ap = addend ? padded(addend->view({T, d}), T, dp) : Tensor();
        if (Yp.defined() && (!addend || ap.defined())) {
          const Tensor full = combine(Yp, gates, k, addend ? Opt(ap) : std::nullopt, out_rows, out_total);
          Tensor out = empty({full.size(0), d}, Y);
          if (copy_pad_into(full, out)) return out;
        }
      }
      const float* g = gates ? ptr<const float>(*gates) : nullptr;
      const void* add = addend ? raw(*addend) : nullptr;
      if (!out_rows) {
        Tensor out = empty({T, d}, Y);
        if (zmoe_combine(raw(Y), g, add, T, (int)k, d, code(Y), raw(out), stream_of(Y)) == ZMOE_OK) return out;
      } else {
        Tensor out = at::zeros({out_total, d}, Y.options());
        if (zmoe_combine_rows(raw(Y), g, add, T, (int)k, d, code(Y), ids(*out_rows), out_total, raw(out),
                              stream_of(Y)) == ZMOE_OK)
          return out;
      }
    }
  }
  static const auto op = general<Tensor(const Tensor&, const Opt&, c10::SymInt, const Opt&, const Opt&, c10::SymInt)>(
      "zmoe::combine");
  return op.call(Y, gates, k, addend, out_rows, out_total);
}

Tensors combine_backward(const Tensor& Y, const Tensor& dout, const Tensor& gates, const Tensor& inv,
                         const Opt& grad_rows) {
  if (Y.is_cuda() && known(Y) && Y.is_contiguous() && flat(dout, Y, Y.scalar_type()) && dout.dim() >= 1 &&
      flat(gates, Y, at::kFloat) && gates.dim() == 2 && flat(inv, Y, at::kInt) && fits_int(gates.size(1))) {
    const int64_t T = gates.size(0), k = gates.size(1), d = dout.size(-1);
    if (inv.numel() == T * k && Y.numel() == T * k * d && d > 0 &&
        (grad_rows ? index(*grad_rows, Y, T) : dout.numel() == T * d)) {
      const c10::DeviceGuard guard(Y.device());
      Tensor dg = empty({T, k}, Y, at::kFloat), grouped = empty({T * k, d}, Y);
      const int rc =
          grad_rows ? zmoe_combine_backward_rows(raw(Y), raw(dout), ids(*grad_rows), dout.numel() / d,
                                                 ptr<const float>(gates), ptr<const int32_t>(inv), T, (int)k, d,
                                                 code(Y), ptr<float>(dg), raw(grouped), stream_of(Y))
                    : zmoe_combine_backward(raw(Y), raw(dout), ptr<const float>(gates), ptr<const int32_t>(inv), T,
                                            (int)k, d, code(Y), ptr<float>(dg), raw(grouped), stream_of(Y));
      if (rc == ZMOE_OK) return {dg, grouped};
    }
  }
  static const auto op = general<Tensors(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Opt&)>(
      "zmoe::combine_backward");
  return op.call(Y, dout, gates, inv, grad_rows);
}

Tensor sum_k(const Tensor& Xe, int64_t k, const Opt& add0, bool out_f32) {
  if (Xe.is_cuda() && known(Xe) && Xe.dim() == 2 && Xe.is_contiguous() && k > 0 && fits_int(k) &&
      Xe.size(0) % k == 0) {
    const int64_t T = Xe.size(0) / k, d = Xe.size(1);
    if (!add0 || (flat(*add0, Xe, Xe.scalar_type()) && add0->numel() == T * d)) {
      const c10::DeviceGuard guard(Xe.device());
      if (const int64_t dp = up(d, Xe); dp != d) {
        const Tensor Xp = padded(Xe, T * k, dp), ap = add0 ? padded(add0->view({T, d}), T, dp) : Tensor();
        if (Xp.defined() && (!add0 || ap.defined())) {
          const Tensor full = sum_k(Xp, k, add0 ? Opt(ap) : std::nullopt, out_f32);
          Tensor out = empty({T, d}, full);
          if (copy_pad_into(full, out)) return out;
        }
      }
      Tensor out = empty({T, d}, Xe, wgrad_dtype(Xe, out_f32));
      if (zmoe_sum_k(raw(Xe), T, (int)k, d, code(Xe), add0 ? raw(*add0) : nullptr, nullptr, code(out), raw(out),
                     stream_of(Xe)) == ZMOE_OK)
        return out;
    }
  }
  static const auto op = general<Tensor(const Tensor&, c10::SymInt, const Opt&, bool)>("zmoe::sum_k");
  return op.call(Xe, k, add0, out_f32);
}

Tensor cast_bf16(const Tensor& src) {
  if (src.is_cuda() && src.scalar_type() == at::kFloat && src.is_contiguous()) {
    const c10::DeviceGuard guard(src.device());
    Tensor out = empty(src.sizes(), src, at::kBFloat16);
    if (zmoe_cast_f32_bf16(ptr<const float>(src), src.numel(), raw(out), stream_of(src)) == ZMOE_OK) return out;
  }
  static const auto op = general<Tensor(const Tensor&)>("zmoe::cast_bf16");
  return op.call(src);
}

Tensors cast_bf16_packed(at::TensorList srcs, int64_t cat_from, int64_t any_from) {
  const int64_t n = (int64_t)srcs.size();
  if (cat_from >= 0 && cat_from < n && n <= ZMOE_CAST_MAX_SEGMENTS && srcs[0].is_cuda()) {
    const Tensor& x = srcs[0];
    bool ok = true;
    int64_t rows = 0;
    for (int64_t i = 0; i < n; ++i) {
      ok = ok && flat(srcs[i], x, at::kFloat) && srcs[i].dim() >= 1;
      if (ok && i >= cat_from) {
        ok = srcs[i].sizes().slice(1) == srcs[cat_from].sizes().slice(1);
        rows += srcs[i].size(0);
      }
    }
    if (ok) {
      const c10::DeviceGuard guard(x.device());
      Tensors out;
      const float* src[ZMOE_CAST_MAX_SEGMENTS];
      int64_t count[ZMOE_CAST_MAX_SEGMENTS];
      void* dst[ZMOE_CAST_MAX_SEGMENTS];
      for (int64_t i = 0; i < cat_from; ++i) out.push_back(empty(srcs[i].sizes(), x, at::kBFloat16));
      auto shape = srcs[cat_from].sizes().vec();
      shape[0] = rows;
      out.push_back(empty(shape, x, at::kBFloat16));
      int64_t at = 0;
      for (int64_t i = 0; i < n; ++i) {
        src[i] = ptr<const float>(srcs[i]);
        count[i] = srcs[i].numel();
        dst[i] = i < cat_from ? raw(out[i]) : static_cast<char*>(raw(out[cat_from])) + 2 * at;
        if (i >= cat_from) at += count[i];
      }
      if (zmoe_cast_f32_bf16_segments(src, count, dst, (int)n, stream_of(x)) == ZMOE_OK) return out;
    }
  }
  static const auto op = general<Tensors(at::TensorList, c10::SymInt, c10::SymInt)>("zmoe::cast_bf16_packed");
  return op.call(srcs, cat_from, any_from);
}

Tensor swiglu(const Tensor& H) {
  if (H.is_cuda() && known(H) && H.dim() == 2 && H.is_contiguous()) {
    const c10::DeviceGuard guard(H.device());
    Tensor A = empty({H.size(0), H.size(1) / 2}, H);
    if (zmoe_swiglu(raw(H), H.size(0), H.size(1) / 2, code(H), raw(A), stream_of(H)) == ZMOE_OK) return A;
  }
  static const auto op = general<Tensor(const Tensor&)>("zmoe::swiglu");
  return op.call(H);
}

Tensor swiglu_backward(const Tensor& dA, const Tensor& H) {
  if (H.is_cuda() && known(H) && H.dim() == 2 && H.is_contiguous() && flat(dA, H, H.scalar_type()) &&
      dA.numel() * 2 == H.numel()) {
    const c10::DeviceGuard guard(H.device());
    Tensor dH = empty(H.sizes(), H);
    if (zmoe_swiglu_backward(raw(dA), raw(H), H.size(0), H.size(1) / 2, code(H), raw(dH), H.size(1), stream_of(H)) ==
        ZMOE_OK)
      return dH;
  }
  static const auto op = general<Tensor(const Tensor&, const Tensor&)>("zmoe::swiglu_backward");
  return op.call(dA, H);
}

Tensors swiglu_backward_gates(const Tensor& dA, const Tensor& H, const Tensor& scale, const Tensor& slots) {
  if (H.is_cuda() && known(H) && H.dim() == 2 && H.is_contiguous() && flat(dA, H, H.scalar_type()) && dA.dim() == 2 &&
      dA.size(0) == H.size(0) && dA.size(1) * 2 == H.size(1) && flat(scale, H, at::kFloat) &&
      scale.numel() == H.size(0) && index(slots, H, H.size(0))) {
    const c10::DeviceGuard guard(H.device());
    Tensor dH = empty(H.sizes(), H), dg = empty({H.size(0)}, H, at::kFloat);
    if (zmoe_swiglu_backward_gates(raw(dA), raw(H), H.size(0), dA.size(1), ptr<const float>(scale), ids(slots),
                                   code(H), raw(dH), ptr<float>(dg), stream_of(H)) == ZMOE_OK)
      return {dH, dg};
  }
  static const auto op = general<Tensors(const Tensor&, const Tensor&, const Tensor&, const Tensor&)>(
      "zmoe::swiglu_backward_gates");
  return op.call(dA, H, scale, slots);
}

Tensors rmsnorm_rows(const Tensor& X, const Tensor& weight, double eps, const Opt& rows) {
  if (X.is_cuda() && known(X) && rows2(X, X) && on(weight, X) && known(weight) && weight.is_contiguous() &&
      weight.numel() == X.size(1) && (!rows || flat(*rows, X, at::kLong))) {
    const c10::DeviceGuard guard(X.device());
    const int64_t N = X.size(0), d = X.size(1), n = rows ? rows->numel() : N;
    Tensor Y = empty({n, d}, X), rstd = empty({n}, X, at::kFloat);
    if (zmoe_rmsnorm_rows(raw(X), X.stride(0), N, rows ? ids(*rows) : nullptr, n, d, raw(weight), code(weight),
                          (float)eps, code(X), raw(Y), ptr<float>(rstd), stream_of(X)) == ZMOE_OK)
      return {Y, rstd};
  }
  static const auto op =
      general<Tensors(const Tensor&, const Tensor&, double, const Opt&)>("zmoe::rmsnorm_rows");
  return op.call(X, weight, eps, rows);
}

Tensors rmsnorm_rows_backward(const Tensor& dY, const Tensor& X, const Opt& rows, const Tensor& rstd,
                              const Tensor& weight) {
  if (X.is_cuda() && known(X) && X.dim() == 2 && X.is_contiguous() && flat(dY, X, X.scalar_type()) && dY.dim() == 2 &&
      on(weight, X) && known(weight) && weight.is_contiguous() && weight.numel() == X.size(1) &&
      (!rows || flat(*rows, X, at::kLong))) {
    const int64_t N = X.size(0), d = X.size(1), n = rows ? rows->numel() : N;
    if (dY.size(0) == n && dY.size(1) == d && flat(rstd, X, at::kFloat) && rstd.numel() == n) {
      const c10::DeviceGuard guard(X.device());
      Tensor dX = rows ? at::zeros({N, d}, X.options()) : empty({N, d}, X);
      Tensor dw = empty(weight.sizes(), weight);
      const size_t bytes = zmoe_rmsnorm_rows_backward_workspace_bytes(n, d, code(X));
      Tensor ws = workspace(bytes, X);
      if (zmoe_rmsnorm_rows_backward(raw(dY), raw(X), d, N, rows ? ids(*rows) : nullptr, n, d, ptr<const float>(rstd),
                                     raw(weight), code(weight), code(X), raw(dX), d, raw(dw), raw(ws), bytes,
                                     stream_of(X)) == ZMOE_OK)
        return {dX, dw};
    }
  }
  static const auto op = general<Tensors(const Tensor&, const Tensor&, const Opt&, const Tensor&, const Tensor&)>(
      "zmoe::rmsnorm_rows_backward");
  return op.call(dY, X, rows, rstd, weight);
}

// ------------------------------------------------------------------ mutating building blocks
void rowwise_sum_product(const Tensor& out, const Tensor& A, const Tensor& B) {
  if (A.is_cuda() && known(A) && A.dim() == 3 && A.is_contiguous() && on(B, A) && known(B) && B.dim() == 2 &&
      B.is_contiguous() && B.size(0) == A.size(0) && B.size(1) == A.size(2) && on(out, A) && known(out) &&
      out.is_contiguous() && out.numel() == A.size(0) * A.size(1) && fits_int(A.size(1))) {
    const c10::DeviceGuard guard(A.device());
    if (zmoe_rowwise_sum_product(raw(A), code(A), raw(B), code(B), A.size(0), (int)A.size(1), A.size(2), raw(out),
                                 code(out), stream_of(A)) == ZMOE_OK)
      return;
  }
  static const auto op = general<void(const Tensor&, const Tensor&, const Tensor&)>("zmoe::rowwise_sum_product");
  op.call(out, A, B);
}

// Y = the grouped rows; false where the general form has to run.
bool group_into(const Tensor& A, const Tensor& Y, const Opt& coeff, bool has_coeff, int64_t fan_out,
                const Tensor& idx) {
  const bool use = has_coeff && coeff;
  if (A.is_cuda() && known(A) && rows2(A, A) && fan_out > 0 && fits_int(fan_out) &&
      index(idx, A, A.size(0) * fan_out) && rows2(Y, A) && Y.size(0) == idx.numel() && Y.size(1) == A.size(1) &&
      (!use || (on(*coeff, A) && known(*coeff) && coeff->is_contiguous() && coeff->numel() == idx.numel()))) {
    const c10::DeviceGuard guard(A.device());
    if (const int64_t Kp = up(A.size(1), A); Kp != A.size(1)) {
      if (!Y.is_contiguous()) return false;
      const Tensor Ap = padded(A, A.size(0), Kp), Yp = empty({Y.size(0), Kp}, Y);
      return Ap.defined() && group_into(Ap, Yp, coeff, has_coeff, fan_out, idx) && copy_pad_into(Yp, Y);
    }
    return zmoe_group(raw(A), A.stride(0), A.size(1), code(A), ids(idx), idx.numel(), (int)fan_out,
                      use ? raw(*coeff) : nullptr, use ? code(*coeff) : ZMOE_DTYPE_F32, raw(Y), Y.stride(0),
                      stream_of(A)) == ZMOE_OK;
  }
  return false;
}

void group(const Tensor& A, int64_t K, int64_t N, const Tensor& Y, const Opt& coeff, bool has_coeff, int64_t fan_out,
           const Tensor& idx) {
  if (group_into(A, Y, coeff, has_coeff, fan_out, idx)) return;
  static const auto op = general<void(const Tensor&, c10::SymInt, c10::SymInt, const Tensor&, const Opt&, bool,
                                      c10::SymInt, const Tensor&)>("zmoe::group");
  op.call(A, K, N, Y, coeff, has_coeff, fan_out, idx);
}

void groupXtY(int64_t E, const Tensor& DW, const Opt& Db, const Tensor& DY, const Tensor& X, const Tensor& off) {
  if (DW.dim() == 3 && DY.is_cuda() && DY.dim() == 2 && X.dim() == 2 && E >= 0) {
    const Tensor DWt = DW.permute({0, 2, 1});
    if (flat(DWt, DY, DY.scalar_type()) && DWt.size(0) == E && DWt.size(1) == DY.size(1) && DWt.size(2) == X.size(1) &&
        (!Db || (flat(*Db, DY, DY.scalar_type()) && Db->dim() == 2 && Db->size(0) == E && Db->size(1) == DY.size(1)))) {
      const c10::DeviceGuard guard(DY.device());
      if (wgrad_into(DY, X, off, E, std::nullopt, 1, DWt, Db)) return;
    }
  }
  static const auto op = general<void(c10::SymInt, const Tensor&, const Opt&, const Tensor&, const Tensor&,
                                      const Tensor&)>("zmoe::groupXtY");
  op.call(E, DW, Db, DY, X, off);
}

}  // namespace

#define ZMOE_EAGER(name, schema) \
  m.def(#name schema);           \
  m.impl(#name, c10::DispatchKey::CompositeExplicitAutograd, TORCH_FN(name))

TORCH_LIBRARY(zmoe_eager, m) {
  ZMOE_EAGER(route_topk, "(Tensor logits, Tensor expert_biases, int k, bool round_probs_bf16) -> Tensor[]");
  ZMOE_EAGER(swiglu_route_backward,
             "(Tensor dAs, Tensor Hs, Tensor d_gates, Tensor topk_prob, Tensor topk_idx, int num_experts) -> Tensor");
  ZMOE_EAGER(route_topk_backward,
             "(Tensor d_weight, Tensor topk_prob, Tensor topk_idx, int num_experts, Tensor like) -> Tensor");
  ZMOE_EAGER(flatten_sort_count, "(Tensor expert_idxs, int num_experts) -> Tensor[]");
  ZMOE_EAGER(flatten_sort_count_weights, "(Tensor expert_idxs, Tensor weights, int num_experts) -> Tensor[]");
  ZMOE_EAGER(glu_shared_forward,
             "(Tensor x, Tensor W1, Tensor W2, Tensor sorted_scattered_idxs, Tensor expert_offsets, int k, "
             "Tensor row_scale, Tensor W_up, Tensor W_gate, Tensor W_down) -> Tensor[]");
  ZMOE_EAGER(glu_w1_forward,
             "(Tensor x, Tensor W1, Tensor sorted_expert_idxs, Tensor sorted_scattered_idxs, Tensor expert_offsets, "
             "int k, Tensor? row_scale) -> Tensor[]");
  ZMOE_EAGER(glu_act_forward,
             "(Tensor x, Tensor W1, Tensor sorted_scattered_idxs, Tensor expert_offsets, int k, Tensor? row_scale) "
             "-> Tensor");
  ZMOE_EAGER(grouped_mm,
             "(Tensor X, Tensor W, Tensor sorted_expert_idxs, Tensor sorted_scattered_idxs, int k, bool x_grouped, "
             "bool y_grouped, Tensor expert_offsets, str region) -> Tensor");
  ZMOE_EAGER(glu_w2_backward_dh,
             "(Tensor dYg, Tensor W2, Tensor H, Tensor sorted_expert_idxs, Tensor expert_offsets) -> Tensor");
  ZMOE_EAGER(group_bwd_w,
             "(Tensor DY, Tensor X, Tensor expert_offsets, int num_experts, Tensor? x_gather, int x_div, "
             "bool out_f32=False) -> Tensor");
  ZMOE_EAGER(group_bwd_w_bias,
             "(Tensor DY, Tensor X, Tensor expert_offsets, int num_experts, Tensor? x_gather, int x_div) -> Tensor[]");
  ZMOE_EAGER(group_bwd_w_gather_dy,
             "(Tensor DY, Tensor dy_gather, int dy_div, Tensor X, Tensor expert_offsets, int num_experts, "
             "bool out_f32=False) -> Tensor");
  ZMOE_EAGER(dense_wgrad, "(Tensor DY, Tensor X, bool out_f32=False) -> Tensor");
  ZMOE_EAGER(combine,
             "(Tensor Y, Tensor? gates, int k, Tensor? addend, Tensor? out_rows, int out_total) -> Tensor");
  ZMOE_EAGER(combine_backward,
             "(Tensor Y, Tensor grad_out, Tensor gates, Tensor inverse, Tensor? grad_rows) -> Tensor[]");
  ZMOE_EAGER(sum_k, "(Tensor Xe, int k, Tensor? add0, bool out_f32=False) -> Tensor");
  ZMOE_EAGER(cast_bf16, "(Tensor src) -> Tensor");
  ZMOE_EAGER(cast_bf16_packed, "(Tensor[] srcs, int cat_from, int any_from=-1) -> Tensor[]");
  ZMOE_EAGER(swiglu, "(Tensor H) -> Tensor");
  ZMOE_EAGER(swiglu_backward, "(Tensor dA, Tensor H) -> Tensor");
  ZMOE_EAGER(swiglu_backward_gates, "(Tensor dA, Tensor H, Tensor row_scale, Tensor slot_of_row) -> Tensor[]");
  ZMOE_EAGER(rmsnorm_rows, "(Tensor X, Tensor weight, float eps, Tensor? rows) -> Tensor[]");
  ZMOE_EAGER(rmsnorm_rows_backward,
             "(Tensor dY, Tensor X, Tensor? rows, Tensor rstd, Tensor weight) -> Tensor[]");
  ZMOE_EAGER(rowwise_sum_product, "(Tensor(a!) output, Tensor A, Tensor B) -> ()");
  ZMOE_EAGER(group,
             "(Tensor A, int K, int N, Tensor(a!) Y, Tensor? coeff, bool has_coeff, int fan_out, "
             "Tensor sorted_expert_idxs) -> ()");
  ZMOE_EAGER(scatter2scatter,
             "(Tensor(a!) output, Tensor W, Tensor X, int k, Tensor sorted_expert_idxs, Tensor sorted_scattered_idxs, "
             "Tensor? b, bool x_grouped, bool y_grouped, Tensor? expert_offsets) -> ()");
  ZMOE_EAGER(groupXtY,
             "(int E, Tensor(a!) DW, Tensor(b!)? Db, Tensor DY, Tensor X, Tensor expert_offsets) -> ()");
}
