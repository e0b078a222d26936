// What a token's latent attention needs between its projections and its queries (include/vmi_hybrid.h: vmi_hy_latent_prep), for the kernels of prompts and of that name and for the
// one that has a product beside it (vmi_hy_latent_in).
#pragma once
#include "hybrid_common.hpp"

namespace vmi_hybrid {

int check_latent_prep(const vmi_hy_latent_prep_args* a, const vmi_hy_step* s, const char* who);   // the code of what does not fit
inline size_t latent_prep_lds(int rot_n) { return (size_t)(4 + rot_n) * 4; }

// RMS norm of the latent, rotation of the shared key and of the query parts; 256 threads a token.  PROMPT: the query parts in place (a thread's pairs are nobody else's), the
// cache row to row t of `rows` too
template <typename T, bool PROMPT>
__device__ __forceinline__ void latent_prep_token(const vmi_hy_latent_prep_args& p, const vmi_hy_step& s, void* const rows, const int t, float* const lds) {
  float* const part = lds;       // [4]
  float* const cs = lds + 4;     // [rot_n / 2][2]
  need(p.proj), need(p.q), need(p.cache), need(p.norm_w), need(p.freq), need(p.ldp), need(p.heads), need(p.dim), need(p.rot), need(p.rank), need(p.rot_n), need(p.rank_n),
      need(p.eps), need(s.tok_seq), need(s.tok_pos), need(s.tok_slot);
  const int tid = threadIdx.x, half = p.rot_n >> 1, hd = p.dim + p.rot, D = p.rank + p.rot;
  const int seq = s.tok_seq[t];
  const int64_t slot = s.tok_slot[t];
  const double pos = (double)s.tok_pos[t];
  const T* row = static_cast<const T*>(p.proj) + (int64_t)t * p.ldp;
  const T* lat = row + p.heads * hd;
  f32x8 v0 = to_f32<T>(load8(lat + min(tid * 8, p.rank - 8))), w0 = load8(p.norm_w + min(tid * 8, p.rank - 8));
  if (seq < 0) return;
  for (int i = tid; i < half; i += 256) {   // the angle reduced in fp64: exact to fp32 at any position
    const double a = pos * p.freq[i];
    const float r = (float)(a - 6.283185307179586476925 * rint(a * 0.15915494309189533577));
    cs[2 * i] = cosf(r);
    cs[2 * i + 1] = sinf(r);
  }
  float ss = 0.f;
  for (int k = tid * 8; k < p.rank; k += 2048) {
    const f32x8 v = k < 2048 ? v0 : to_f32<T>(load8(lat + k));
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  const float rms = 1.f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)p.rank_n + p.eps);
  T* crow = slot >= 0 ? static_cast<T*>(p.cache) + slot * D : nullptr;
  T* prow = PROMPT ? static_cast<T*>(rows) + (int64_t)t * D : nullptr;
  if (crow || PROMPT) {
    for (int k = tid * 8; k < p.rank; k += 2048) {
      f32x8 v = k < 2048 ? v0 : to_f32<T>(load8(lat + k));
      const f32x8 w = k < 2048 ? w0 : load8(p.norm_w + k);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * rms * w[e];
      if (crow) *reinterpret_cast<V8<T>*>(crow + k) = from_f32<T>(v);
      if constexpr (PROMPT) *reinterpret_cast<V8<T>*>(prow + k) = from_f32<T>(v);
    }
  }
  if (PROMPT || (half & 7) == 0) {   // eight pairs at a time
    const int per = half >> 3;
    for (int u = tid; u < (p.heads + 1) * per; u += 256) {
      const int h = u / per, i = (u - h * per) * 8;
      const T* src = h < p.heads ? row + h * hd + p.dim : lat + p.rank;
      T* dst = h < p.heads ? (PROMPT ? const_cast<T*>(src) : static_cast<T*>(p.q) + ((int64_t)t * p.heads + h) * D + p.rank) : (crow ? crow + p.rank : nullptr);
      T* const second = PROMPT && h == p.heads ? prow + p.rank : nullptr;
      if (!dst && !second) continue;
      const f32x8 a = to_f32<T>(load8(src + i)), b = to_f32<T>(load8(src + i + half));
      f32x8 x, y;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float c = cs[2 * (i + e)], sn = cs[2 * (i + e) + 1];
        x[e] = a[e] * c - b[e] * sn;
        y[e] = b[e] * c + a[e] * sn;
      }
      auto put = [&](T* to) {
        *reinterpret_cast<V8<T>*>(to + i) = from_f32<T>(x);
        *reinterpret_cast<V8<T>*>(to + i + half) = from_f32<T>(y);
        if (i == 0 && to != src)
          for (int k = p.rot_n; k < p.rot; k += 8) *reinterpret_cast<V8<T>*>(to + k) = load8(src + k);   // passes unrotated
      };
      if (dst) put(dst);
      if (second) put(second);
    }
    return;
  }
  if constexpr (PROMPT) return;
  // heads 0 .. heads - 1: the query's rotated part; "head" `heads`: the shared key
  T* qrow = static_cast<T*>(p.q) + (int64_t)t * p.heads * D;
  for (int u = tid; u < (p.heads + 1) * p.rot; u += 256) {
    const int h = u / p.rot, i = u - h * p.rot;
    const T* src = h < p.heads ? row + h * hd + p.dim : lat + p.rank;
    T* dst = h < p.heads ? qrow + (int64_t)h * D + p.rank : (crow ? crow + p.rank : nullptr);
    if (!dst) continue;
    if (i >= p.rot_n) {
      dst[i] = src[i];   // passes unrotated (padding: zeros)
    } else if (i < half) {
      dst[i] = (T)((float)src[i] * cs[2 * i] - (float)src[i + half] * cs[2 * i + 1]);
    } else {
      const int j = i - half;
      dst[i] = (T)((float)src[i] * cs[2 * j] + (float)src[j] * cs[2 * j + 1]);
    }
  }
}

// Entries for latent_prompt_kernel, `rows` beginning at token row0: all, or, mixed, those without a past, and the others as they are without it
__device__ __forceinline__ void latent_prompt_prep_token(const vmi_hy_latent_prep_args& p, const vmi_hy_step& s, b16* const rows, const int row0, const bool mixed, const int t,
                                                         float* const lds) {
  const int e = s.tok_seq[t];
  if (e < 0) return;
  if (!mixed || s.ctx[e] == 0) latent_prep_token<b16, true>(p, s, rows - (int64_t)row0 * (p.rank + p.rot), t, lds);   // (workgroup-uniform)
  else latent_prep_token<b16, false>(p, s, nullptr, t, lds);
}

int check_latent_prompt_prep(const vmi_hy_latent_prep_args* a, const void* rows, int row0, bool mixed, const vmi_hy_step* s, const char* who);
int launch_latent_prompt_prep(const vmi_hy_latent_prep_args& a, void* rows, int row0, bool mixed, const vmi_hy_step& s, hipStream_t st, const char* who);
// ... and l, the other entries' queries by heads into a's q, which does not read what that writes nor writes what it reads: few rows in one launch
int launch_latent_prompt_in(const vmi_hy_linear_args& l, const vmi_hy_latent_prep_args& a, void* rows, int row0, bool mixed, const vmi_hy_step& s, hipStream_t st, const char* who);

}  // namespace vmi_hybrid
