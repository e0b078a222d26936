// What the linear layers' units share: the way out of a product, and the kernels for few rows that hybrid_rows.hip holds.
#pragma once

#include "hybrid_common.hpp"

namespace vmi_hybrid {

// Four consecutive columns n .. n + 3 of row m, accumulated, on their way out.  n0: the first column of their tile (scalar)
template <typename T, int EPI>
__device__ __forceinline__ void epilogue(const vmi_hy_linear_args& p, const f32x4& acc, int m, int n, int n0, int grp) {
  const int64_t yoff = (int64_t)m * p.ldy + (int64_t)grp * p.y_gstride;
  if constexpr (EPI == VMI_HY_E_STORE) {
    f32x4 b = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.bias) b = *reinterpret_cast<const f32x4*>(p.bias + n);
    V4<T> o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (T)(acc[r] + b[r]);
    *reinterpret_cast<V4<T>*>(static_cast<T*>(p.y) + yoff + n) = o;
  } else if constexpr (EPI == VMI_HY_E_RESIDUAL) {
    f32x4* y = reinterpret_cast<f32x4*>(static_cast<float*>(p.y) + yoff + n);
    *y = *y + acc;
  } else if constexpr (EPI == VMI_HY_E_FLOAT) {
    float* y = static_cast<float*>(p.y) + yoff + n;
    if (n + 4 <= p.n_out && (p.ldy & 3) == 0) {
      *reinterpret_cast<f32x4*>(y) = acc * p.scale;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < p.n_out) y[r] = acc[r] * p.scale;
    }
  } else if constexpr (EPI == VMI_HY_E_GLU) {
    typename Elem<T>::v2 o;
    o[0] = (T)glu(acc[0], acc[1], p.scale, p.glu_alpha, p.glu_up);
    o[1] = (T)glu(acc[2], acc[3], p.scale, p.glu_alpha, p.glu_up);
    *reinterpret_cast<typename Elem<T>::v2*>(static_cast<T*>(p.y) + yoff + (n >> 1)) = o;
  } else if constexpr (EPI == VMI_HY_E_STORE_GLU) {
    if (n0 < p.n_split) {
      V4<T> o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (T)acc[r];
      *reinterpret_cast<V4<T>*>(static_cast<T*>(p.y) + yoff + n) = o;
    } else {
      typename Elem<T>::v2 o;
      o[0] = (T)glu(acc[0], acc[1], p.scale, p.glu_alpha, p.glu_up);
      o[1] = (T)glu(acc[2], acc[3], p.scale, p.glu_alpha, p.glu_up);
      *reinterpret_cast<typename Elem<T>::v2*>(static_cast<T*>(p.y2) + (int64_t)m * p.ldy2 + ((n - p.n_split) >> 1)) = o;
    }
  } else {   // VMI_HY_E_GATED
    const float g = sigmoid((float)static_cast<const T*>(p.gate)[(int64_t)m * p.ldg + grp]);
    V4<T> o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (T)(acc[r] * g);
    *reinterpret_cast<V4<T>*>(static_cast<T*>(p.y) + yoff + n) = o;
  }
}

// Products of few rows in bfloat16 (hybrid_rows.hip).  Each is built for what its rule names
int norm_slabs(int M, int N, int K);   // behind a norm, one group: 0 where it is not
int launch_norm_rows(const vmi_hy_linear_args& p, hipStream_t st);
bool held_rows_pay(int M, int N, int K, bool stored);   // of the element type behind a norm of their own, one group; stored: as they are
int launch_held_rows(const vmi_hy_linear_args& p, hipStream_t st);
int check_linear(const vmi_hy_linear_args* a, const char* who);   // the code of what does not fit
bool plain_rows_fit(int M, int N, int K, int groups);   // of the element type
int launch_plain_rows(const vmi_hy_linear_args& p, hipStream_t st);
bool concat_rows_fit(int M, int N, int K);   // float32 rows side by side, FLOAT, one group
int launch_concat_rows(const vmi_hy_linear_args& p, hipStream_t st);
bool group_tiles_fit(const vmi_hy_linear_args& p);   // STORE or GATED, of the element type, many rows (hybrid_tiles.hip)
int launch_group_tiles(const vmi_hy_linear_args& p, hipStream_t st);
int launch_norm_few(const vmi_hy_linear_args& p, hipStream_t st);   // p.normed = the norm of p.x

}  // namespace vmi_hybrid
