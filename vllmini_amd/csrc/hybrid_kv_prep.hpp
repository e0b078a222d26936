// What a token's grouped attention needs between its projections and its queries (include/vmi_hybrid.h: vmi_hy_kv_prep), for the kernel of that name and for the one that has a
// product beside it (vmi_hy_kv_prep_in).
#pragma once
#include "hybrid_softmax.hpp"

namespace vmi_hybrid {

int check_kv_prep(const vmi_hy_kv_prep_args* a, const vmi_hy_step* s, const char* who);   // the code of what does not fit

// q and k over their root mean square, k and v into the cache; 256 threads a token, 16 lanes a head
template <typename T>
__device__ __forceinline__ void kv_prep_token(const vmi_hy_kv_prep_args& p, const vmi_hy_step& s, const int t) {
  const int tid = threadIdx.x, l = tid & 15, D = p.dim + p.vdim;
  if (s.tok_seq[t] < 0) return;
  const int64_t slot = s.tok_slot[t];
  const T* row = static_cast<const T*>(p.proj) + (int64_t)t * p.ldp;
  T* crow = slot >= 0 ? static_cast<T*>(p.cache) + slot * p.kv_heads * D : nullptr;
  for (int u = tid >> 4; u < p.heads + p.kv_heads; u += 16) {
    const T* src = row + (int64_t)u * p.dim;
    float ss = 0.f;
    for (int k = l * 8; k < p.dim; k += 128) {
      const f32x8 v = to_f32<T>(load8(src + k));
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
    }
    ss = sum16(ss);
    const float r = 1.f / sqrtf(ss / (float)p.dim_n + p.eps);
    T* dst = u < p.heads ? static_cast<T*>(p.q) + ((int64_t)t * p.heads + u) * p.dim : crow ? crow + (int64_t)(u - p.heads) * D : nullptr;
    if (!dst) continue;
    for (int k = l * 8; k < p.dim; k += 128) {
      f32x8 v = to_f32<T>(load8(src + k));
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= r;
      *reinterpret_cast<V8<T>*>(dst + k) = from_f32<T>(v);
    }
  }
  if (!crow) return;
  const T* v = row + (int64_t)(p.heads + p.kv_heads) * p.dim;
  for (int u = tid * 8; u < p.kv_heads * p.vdim; u += 2048) {
    const int g = u / p.vdim, k = u - g * p.vdim;
    *reinterpret_cast<V8<T>*>(crow + (int64_t)g * D + p.dim + k) = load8(v + u);
  }
}

}  // namespace vmi_hybrid
