// ZeroCenteredRMSNorm (modeling/zRMSNorm.py:10-17) fused with the unpad gather in front of
// the MoE layer (modeling/moe_layer.py:39-42, flash_attn's index_first_axis):
//   Y[i] = X[rows[i]] * rsqrt(mean(X[rows[i]]^2) + eps) * (1 + w)      (fp32, stored as X's dtype)
// one pass that reads each selected row once, and its backward
//   dX[rows[i]] = r (1 + w) dy - X r^3 / d * sum_j dy_j (1 + w_j) X_j     (r = the saved rstd)
//   dw          = sum_i dy_i * X[rows[i]] * r_i                           (fixed-order, deterministic)
// Layout: a row of up to 256 16-byte chunks is one wave's (1, 2 or 4 chunks per lane, the row
// sum a wave reduction, no barrier); a longer one belongs to the four waves of a block (2, 4 or
// 8 chunks per thread, the row sum through LDS). Both passes are bound by HBM: what they need is
// enough rows in flight per CU, so the chunk count is a template parameter (no registers for
// chunks a row does not have) and the backward loads its next row before it reduces the current
// one. At [16383, 2048] bf16: forward 30.6 us (4.4 TB/s; a device copy reaches 4.96), backward
// 35.0 us (5.8 TB/s, reads twice its writes). A block per row with room for 8 chunks in every
// thread, two barriers a row and no prefetch took 31.9 and 70.7 us.
#include <type_traits>

#include "zmoe_internal.h"

namespace zmoe {

constexpr int kNormThreads = 256;
constexpr int kNormWaves = kNormThreads / 64;
constexpr int kNormMaxChunks = 8;
constexpr int kNormMaxPartials = 512;

// Waves per row and 16-byte chunks per thread for rows of nch chunks.
struct NormMap {
  int wpr, nq;
  int rpb() const { return kNormWaves / wpr; }
};

inline NormMap norm_map(int64_t nch) {
  if (nch <= 256) return NormMap{1, nch <= 64 ? 1 : (nch <= 128 ? 2 : 4)};
  return NormMap{4, nch <= 512 ? 2 : (nch <= 1024 ? 4 : 8)};
}

// 1 + w for the VN weights from column c (16-byte loads where the weight's base allows it).
template <int VN, typename TW>
__device__ __forceinline__ void load_gain(const TW* __restrict__ w, int64_t c, bool vec, float (&g)[VN]) {
  constexpr int VW = 16 / sizeof(TW);
  if (vec && VN >= VW) {
#pragma unroll
    for (int q = 0; q < VN / VW; ++q)
      unpack_chunk(*reinterpret_cast<const uint4*>(w + c + q * VW), &g[q * VW], TW{});
  } else {
#pragma unroll
    for (int u = 0; u < VN; ++u) g[u] = to_f32(w[c + u]);
  }
#pragma unroll
  for (int u = 0; u < VN; ++u) g[u] += 1.0f;
}

// Sum of v over the threads of one row. With four waves per row every thread of the block has to
// call it, alternating `parity` between calls (one barrier: a call's LDS slots are read before
// the call after the next one writes them).
template <int WPR>
__device__ __forceinline__ float row_sum(float v, float (&red)[2][kNormWaves], int parity) {
  v = wave_sum(v);
  if constexpr (WPR == 1) {
    return v;
  } else {
    if ((threadIdx.x & 63) == 0) red[parity][threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < kNormWaves; ++q) t += red[parity][q];
    return t;
  }
}

template <typename T, typename TW, int WPR, int NQ>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_rows_kernel(const T* __restrict__ X, int64_t ldx,
                                                                    int64_t x_rows, const int64_t* __restrict__ rows,
                                                                    int64_t n, int64_t d, const TW* __restrict__ w,
                                                                    int w_vec, float eps, T* __restrict__ Y,
                                                                    float* __restrict__ rstd) {
  constexpr int VN = 16 / sizeof(T);
  constexpr int TPR = 64 * WPR;
  __shared__ float red[2][kNormWaves];
  const int64_t i = (int64_t)blockIdx.x * (kNormWaves / WPR) + threadIdx.x / TPR;
  const int lt = threadIdx.x % TPR;
  const int nch = (int)(d / VN);
  int64_t src = -1;
  if (i < n) {
    src = rows ? rows[i] : i;
    if (src < 0 || src >= x_rows) src = -1;  // out-of-range row: written as zeros
  }
  uint4 c[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int ch = lt + q * TPR;
    c[q] = make_uint4(0, 0, 0, 0);
    if (src >= 0 && ch < nch) c[q] = *reinterpret_cast<const uint4*>(X + src * ldx + (int64_t)ch * VN);
  }
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    float v[VN];
    unpack_chunk(c[q], v, T{});
#pragma unroll
    for (int u = 0; u < VN; ++u) ss = fmaf(v[u], v[u], ss);
  }
  const float tot = row_sum<WPR>(ss, red, 0);  // every thread of the block gets here
  if (i >= n) return;
  const float r = src >= 0 ? rsqrtf(tot / (float)d + eps) : 0.f;
  if (rstd && lt == 0) rstd[i] = r;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int ch = lt + q * TPR;
    if (ch < nch) {
      float v[VN], g[VN];
      unpack_chunk(c[q], v, T{});
      load_gain<VN>(w, (int64_t)ch * VN, w_vec != 0, g);
#pragma unroll
      for (int u = 0; u < VN; ++u) v[u] = (v[u] * r) * g[u];
      *reinterpret_cast<uint4*>(Y + i * d + (int64_t)ch * VN) = pack_chunk(v, T{});
    }
  }
}

// One row's operands of the backward: the chunks of X and dY this thread holds.
template <typename T, int NQ>
struct NormRow {
  uint4 x[NQ], g[NQ];
  int64_t src;
  float r;

  template <int TPR>
  __device__ __forceinline__ void load(const T* dY, const T* X, int64_t ldx, int64_t x_rows, const int64_t* rows,
                                       int64_t i, int64_t n, int64_t d, const float* rstd, int lt, int nch) {
    constexpr int VN = 16 / sizeof(T);
    src = -1;
    r = 0.f;
    if (i < n) {
      src = rows ? rows[i] : i;
      if (src < 0 || src >= x_rows) src = -1;
      r = rstd[i];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int ch = lt + q * TPR;
      x[q] = make_uint4(0, 0, 0, 0);
      g[q] = make_uint4(0, 0, 0, 0);
      if (src >= 0 && ch < nch) {
        x[q] = *reinterpret_cast<const uint4*>(X + src * ldx + (int64_t)ch * VN);
        g[q] = *reinterpret_cast<const uint4*>(dY + i * d + (int64_t)ch * VN);
      }
    }
  }
};

// One block per partial: grid-stride over rows, every thread accumulating dw for its own columns
// in registers; with one wave per row the block's four sums are added in wave order through LDS.
template <typename T, typename TW, int WPR, int NQ>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_rows_backward_kernel(
    const T* __restrict__ dY, const T* __restrict__ X, int64_t ldx, int64_t x_rows, const int64_t* __restrict__ rows,
    int64_t n, int64_t d, const float* __restrict__ rstd, const TW* __restrict__ w, int w_vec, T* __restrict__ dX,
    int64_t lddx, float* __restrict__ partial) {
  constexpr int VN = 16 / sizeof(T);
  constexpr int TPR = 64 * WPR, RPB = kNormWaves / WPR;
  constexpr bool PREFETCH = NQ <= 4;  // at 8 chunks the next row's registers do not fit
  extern __shared__ float slot_dw[];  // WPR == 1: [RPB][d]
  __shared__ float red[2][kNormWaves];
  const int slot = threadIdx.x / TPR, lt = threadIdx.x % TPR;
  const int nch = (int)(d / VN);
  float acc[NQ][VN], gain[NQ][VN];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
#pragma unroll
    for (int u = 0; u < VN; ++u) acc[q][u] = gain[q][u] = 0.f;
    if (lt + q * TPR < nch) load_gain<VN>(w, (int64_t)(lt + q * TPR) * VN, w_vec != 0, gain[q]);
  }
  const float inv_d = 1.0f / (float)d;
  const int64_t step = (int64_t)gridDim.x * RPB;
  const int64_t first = (int64_t)blockIdx.x * RPB;
  int64_t i = first + slot;
  NormRow<T, NQ> cur, nxt;
  cur.template load<TPR>(dY, X, ldx, x_rows, rows, i, n, d, rstd, lt, nch);
  int parity = 0;
  for (int64_t base = first; base < n; base += step, i += step, parity ^= 1) {  // uniform in the block
    if constexpr (PREFETCH) nxt.template load<TPR>(dY, X, ldx, x_rows, rows, i + step, n, d, rstd, lt, nch);
    float dot = 0.f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      float xv[VN], gv[VN];
      unpack_chunk(cur.x[q], xv, T{});
      unpack_chunk(cur.g[q], gv, T{});
#pragma unroll
      for (int u = 0; u < VN; ++u) {
        dot = fmaf(gv[u] * gain[q][u], xv[u], dot);
        acc[q][u] = fmaf(gv[u] * xv[u], cur.r, acc[q][u]);
      }
    }
    const float tot = row_sum<WPR>(dot, red, parity);
    if (cur.src >= 0) {
      const float coef = cur.r * cur.r * cur.r * tot * inv_d;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int ch = lt + q * TPR;
        if (ch < nch) {
          float xv[VN], gv[VN];
          unpack_chunk(cur.x[q], xv, T{});
          unpack_chunk(cur.g[q], gv, T{});
#pragma unroll
          for (int u = 0; u < VN; ++u) gv[u] = cur.r * gv[u] * gain[q][u] - xv[u] * coef;
          *reinterpret_cast<uint4*>(dX + cur.src * lddx + (int64_t)ch * VN) = pack_chunk(gv, T{});
        }
      }
    }
    if constexpr (PREFETCH) cur = nxt;
    else cur.template load<TPR>(dY, X, ldx, x_rows, rows, i + step, n, d, rstd, lt, nch);
  }
  float* dst = RPB == 1 ? partial + (int64_t)blockIdx.x * d : slot_dw + (int64_t)slot * d;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int ch = lt + q * TPR;
    if (ch < nch)
#pragma unroll
      for (int u = 0; u < VN; ++u) dst[(int64_t)ch * VN + u] = acc[q][u];
  }
  if constexpr (RPB == 1) return;
  __syncthreads();
  for (int64_t col = threadIdx.x; col < d; col += kNormThreads) {
    float t = 0.f;
#pragma unroll
    for (int s2 = 0; s2 < RPB; ++s2) t += slot_dw[(int64_t)s2 * d + col];
    partial[(int64_t)blockIdx.x * d + col] = t;
  }
}

// dw[c] = sum over the P partials of partial[p][c], rounded once to the weight's dtype: a block
// takes 64 columns, wave v sums partials v, v + 16, ... and the 16 sums are added in wave order
// (a fixed order, whatever the schedule). Bound by the latency of the partials' loads: at P = 512,
// d = 2048 it takes 4.0 us; one thread per column over all partials (8 blocks) took 118 us.
constexpr int kDwWaves = 16;
template <typename TW>
__global__ __launch_bounds__(64 * kDwWaves) void rmsnorm_dw_reduce_kernel(const float* __restrict__ partial, int P,
                                                                          int64_t d, TW* __restrict__ dw) {
  __shared__ float red[kDwWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t c = (int64_t)blockIdx.x * 64 + lane;
  float t = 0.f;
  if (c < d) {
#pragma unroll 8
    for (int p = wave; p < P; p += kDwWaves) t += partial[(int64_t)p * d + c];
  }
  red[wave][lane] = t;
  __syncthreads();
  if (wave != 0 || c >= d) return;
#pragma unroll
  for (int v = 1; v < kDwWaves; ++v) t += red[v][lane];
  dw[c] = from_f32<TW>(t);
}

int norm_partials(int64_t n, int rpb) {
  const int64_t want = cdiv(n > 0 ? n : 1, rpb);
  return (int)(want < kNormMaxPartials ? want : kNormMaxPartials);
}

// Calls f with the map's waves per row and chunks per thread as compile-time constants.
template <typename F>
void with_norm_map(const NormMap& m, F f) {
  using std::integral_constant;
  if (m.wpr == 1) {
    if (m.nq == 1) f(integral_constant<int, 1>{}, integral_constant<int, 1>{});
    else if (m.nq == 2) f(integral_constant<int, 1>{}, integral_constant<int, 2>{});
    else f(integral_constant<int, 1>{}, integral_constant<int, 4>{});
  } else {
    if (m.nq == 2) f(integral_constant<int, 4>{}, integral_constant<int, 2>{});
    else if (m.nq == 4) f(integral_constant<int, 4>{}, integral_constant<int, 4>{});
    else f(integral_constant<int, 4>{}, integral_constant<int, 8>{});
  }
}

template <typename T, typename TW>
int launch_norm_fwd(const void* X, int64_t ldx, int64_t x_rows, const int64_t* rows, int64_t n, int64_t d,
                    const void* w, float eps, void* Y, float* rstd, hipStream_t s) {
  const NormMap m = norm_map(d / (16 / (int64_t)sizeof(T)));
  with_norm_map(m, [&](auto wpr, auto nq) {
    hipLaunchKernelGGL((rmsnorm_rows_kernel<T, TW, wpr(), nq()>), dim3((unsigned)cdiv(n, m.rpb())),
                       dim3(kNormThreads), 0, s, static_cast<const T*>(X), ldx, x_rows, rows, n, d,
                       static_cast<const TW*>(w), (int)aligned16(w), eps, static_cast<T*>(Y), rstd);
  });
  return check_launch("rmsnorm_rows");
}

template <typename T, typename TW>
int launch_norm_bwd(const void* dY, const void* X, int64_t ldx, int64_t x_rows, const int64_t* rows, int64_t n,
                    int64_t d, const float* rstd, const void* w, void* dX, int64_t lddx, void* dw, float* partial,
                    hipStream_t s) {
  const NormMap m = norm_map(d / (16 / (int64_t)sizeof(T)));
  const int P = norm_partials(n, m.rpb());
  const size_t lds = m.rpb() == 1 ? 0 : (size_t)m.rpb() * (size_t)d * sizeof(float);  // at most 32 KB
  with_norm_map(m, [&](auto wpr, auto nq) {
    hipLaunchKernelGGL((rmsnorm_rows_backward_kernel<T, TW, wpr(), nq()>), dim3((unsigned)P), dim3(kNormThreads), lds,
                       s, static_cast<const T*>(dY), static_cast<const T*>(X), ldx, x_rows, rows, n, d, rstd,
                       static_cast<const TW*>(w), (int)aligned16(w), static_cast<T*>(dX), lddx, partial);
  });
  int rc = check_launch("rmsnorm_rows_backward");
  if (rc) return rc;
  hipLaunchKernelGGL((rmsnorm_dw_reduce_kernel<TW>), dim3((unsigned)cdiv(d, 64)), dim3(64 * kDwWaves), 0, s, partial,
                     P, d, static_cast<TW*>(dw));
  return check_launch("rmsnorm_rows_backward dw");
}

int norm_shape_checks(int64_t x_stride, int64_t x_rows, int64_t n, int64_t d, int w_dtype, int dtype,
                      const char* name) {
  ZMOE_REQUIRE(dtype_ok(dtype) && dtype_ok(w_dtype), ZMOE_ERR_DTYPE, "%s: dtype %d / weight dtype %d", name, dtype,
               w_dtype);
  const int64_t vec = 16 / dtype_size(dtype);
  ZMOE_REQUIRE(n >= 0 && x_rows >= 0 && d >= 1, ZMOE_ERR_SHAPE, "%s: bad sizes (n=%lld d=%lld)", name,
               (long long)n, (long long)d);
  ZMOE_REQUIRE(d <= 256 * kNormMaxChunks * vec, ZMOE_ERR_SHAPE, "%s: d=%lld above the row kernel's %lld", name,
               (long long)d, (long long)(256 * kNormMaxChunks * vec));
  ZMOE_REQUIRE(d % vec == 0 && x_stride % vec == 0 && x_stride >= d, ZMOE_ERR_ALIGN,
               "%s: d and the row stride must be multiples of %lld elements", name, (long long)vec);
  return ZMOE_OK;
}

}  // namespace zmoe

using namespace zmoe;

extern "C" int zmoe_rmsnorm_rows(const void* X, int64_t x_stride, int64_t x_rows, const int64_t* rows, int64_t n,
                                 int64_t d, const void* weight, int w_dtype, float eps, int dtype, void* Y,
                                 float* rstd, void* stream) {
  int rc = norm_shape_checks(x_stride, x_rows, n, d, w_dtype, dtype, "rmsnorm_rows");
  if (rc) return rc;
  if (n == 0) return ZMOE_OK;
  ZMOE_REQUIRE(X && weight && Y, ZMOE_ERR_NULL, "rmsnorm_rows: null pointer");
  ZMOE_REQUIRE(aligned16(X) && aligned16(Y), ZMOE_ERR_ALIGN, "rmsnorm_rows: X and Y must be 16-byte aligned");
  hipStream_t s = as_stream(stream);
  if (dtype == ZMOE_DTYPE_BF16)
    return w_dtype == ZMOE_DTYPE_BF16
               ? launch_norm_fwd<uint16_t, uint16_t>(X, x_stride, x_rows, rows, n, d, weight, eps, Y, rstd, s)
               : launch_norm_fwd<uint16_t, float>(X, x_stride, x_rows, rows, n, d, weight, eps, Y, rstd, s);
  return w_dtype == ZMOE_DTYPE_BF16
             ? launch_norm_fwd<float, uint16_t>(X, x_stride, x_rows, rows, n, d, weight, eps, Y, rstd, s)
             : launch_norm_fwd<float, float>(X, x_stride, x_rows, rows, n, d, weight, eps, Y, rstd, s);
}

extern "C" size_t zmoe_rmsnorm_rows_backward_workspace_bytes(int64_t n, int64_t d, int dtype) {
  if (d < 1 || !dtype_ok(dtype)) return 0;
  const NormMap m = norm_map(d / (16 / dtype_size(dtype)));
  return (size_t)norm_partials(n, m.rpb()) * (size_t)d * sizeof(float);
}

extern "C" int zmoe_rmsnorm_rows_backward(const void* dY, const void* X, int64_t x_stride, int64_t x_rows,
                                          const int64_t* rows, int64_t n, int64_t d, const float* rstd,
                                          const void* weight, int w_dtype, int dtype, void* dX, int64_t dx_stride,
                                          void* dweight, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = norm_shape_checks(x_stride, x_rows, n, d, w_dtype, dtype, "rmsnorm_rows_backward");
  if (rc) return rc;
  const int64_t vec = 16 / dtype_size(dtype);
  ZMOE_REQUIRE(dx_stride % vec == 0 && dx_stride >= d, ZMOE_ERR_ALIGN,
               "rmsnorm_rows_backward: dX row stride must be a multiple of %lld elements", (long long)vec);
  ZMOE_REQUIRE(weight && dweight && workspace, ZMOE_ERR_NULL, "rmsnorm_rows_backward: null pointer");
  ZMOE_REQUIRE(n == 0 || (dY && X && rstd && dX), ZMOE_ERR_NULL, "rmsnorm_rows_backward: null operand");
  const size_t need = zmoe_rmsnorm_rows_backward_workspace_bytes(n, d, dtype);
  ZMOE_REQUIRE(workspace_bytes >= need, ZMOE_ERR_WORKSPACE, "rmsnorm_rows_backward: workspace %zu < %zu bytes",
               workspace_bytes, need);
  ZMOE_REQUIRE((n == 0 || (aligned16(dY) && aligned16(X) && aligned16(dX))) && aligned16(workspace), ZMOE_ERR_ALIGN,
               "rmsnorm_rows_backward: operands must be 16-byte aligned");
  hipStream_t s = as_stream(stream);
  float* partial = static_cast<float*>(workspace);
  if (dtype == ZMOE_DTYPE_BF16)
    return w_dtype == ZMOE_DTYPE_BF16
               ? launch_norm_bwd<uint16_t, uint16_t>(dY, X, x_stride, x_rows, rows, n, d, rstd, weight, dX, dx_stride,
                                                     dweight, partial, s)
               : launch_norm_bwd<uint16_t, float>(dY, X, x_stride, x_rows, rows, n, d, rstd, weight, dX, dx_stride,
                                                  dweight, partial, s);
  return w_dtype == ZMOE_DTYPE_BF16
             ? launch_norm_bwd<float, uint16_t>(dY, X, x_stride, x_rows, rows, n, d, rstd, weight, dX, dx_stride,
                                                dweight, partial, s)
             : launch_norm_bwd<float, float>(dY, X, x_stride, x_rows, rows, n, d, rstd, weight, dX, dx_stride,
                                             dweight, partial, s);
}
