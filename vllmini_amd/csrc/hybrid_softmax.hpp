// Pieces of the softmax attention kernels (hybrid_latent.hip, hybrid_attention.hip): reading an LDS tile by columns, reductions over
// the 16 lanes of a row, and the sum over key splits.
#pragma once
#include "hybrid_common.hpp"

namespace vmi_hybrid {

typedef short s16x4 __attribute__((ext_vector_type(4)));

// 8 consecutive rows (keys) of one column of an LDS tile, as a matrix operand's fragment: lane = (kc, column r16)
__device__ __forceinline__ b16x8 column8(const b16* tile, int ld, int row0, int col0, int r16) {
  const b16* a = tile + (row0 + (r16 >> 2)) * ld + col0 + 4 * (r16 & 3);
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)a);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(a + 4 * ld));
  // (whole vectors are cast: a bit_cast of one vector element takes element 0 on this compiler)
  return __builtin_shufflevector(__builtin_bit_cast(b16x4, lo), __builtin_bit_cast(b16x4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ f32x8 column8(const float* tile, int ld, int row0, int col0, int r16) {
  f32x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = tile[(row0 + e) * ld + col0 + r16];
  return r;
}

// maximum / sum over the 16 lanes that share kc, on the cross-lane paths of the vector unit (no LDS round trip)
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float max16(float v) {
  v = fmaxf(v, dpp<0xB1>(v));    // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp<0x4E>(v));    // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp<0x141>(v));   // row_half_mirror
  return fmaxf(v, dpp<0x140>(v));   // row_mirror
}
__device__ __forceinline__ float sum16(float v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  return v + dpp<0x140>(v);
}

__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

template <typename T>
constexpr int pad_of() {
  return 16 / (int)sizeof(T);
}

struct Combine {
  const float* partial;    // [splits][T * heads][width + 2]: unnormalised sums, their maximum (log2 units), their weight
  void* out;               // [T][ldo], head h at column h * width
  const void* gate;        // [T][ldg] one column per head, or NULL
  const int32_t* tok_seq;
  int64_t ldo, ldg;
  int T, heads, width, splits;
};

// out[row] = sum over splits of 2^(m_s - m) part_s / sum of 2^(m_s - m) l_s (times sigmoid(gate)); one workgroup per (token, head), two columns a thread.  Bound by its
// trips through memory: AHEAD parts are asked for beside their weights, and the following ones AHEAD at a time, all of them without a condition (parts past the last are
// that one again, with a weight of zero): a condition a part waits for each of them.
template <typename T, int AHEAD>
__global__ __launch_bounds__(512) void combine_kernel(const Combine p) {
  need(p.partial), need(p.out), need(p.gate), need(p.tok_seq), need(p.ldo), need(p.ldg), need(p.T), need(p.heads), need(p.width), need(p.splits);
  static_assert(128 % AHEAD == 0, "the weights end with a group of parts");
  const int t = (int)(blockIdx.x / (unsigned)p.heads), h = (int)(blockIdx.x - (unsigned)t * p.heads), seq = p.tok_seq[t];
  const int ld = p.width + 2;
  __shared__ float wt[128];   // weight of every part (at most 128 of them), zeros behind them
  const char* first = reinterpret_cast<const char*>(p.partial + (int64_t)blockIdx.x * ld);
  const int64_t each = (int64_t)p.T * p.heads * ld * 4;
  auto ask = [&](f32x2(&v)[AHEAD], int i0, int k) {
    const uint32_t at = (uint32_t)min(k, p.width - 2) * 4;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) v[i] = *reinterpret_cast<const f32x2*>(first + min(i0 + i, p.splits - 1) * each + at);
  };
  auto ask_weights = [&](int i) { return *reinterpret_cast<const f32x2*>(first + min((int)(threadIdx.x & 63) + i, p.splits - 1) * each + (uint32_t)p.width * 4); };
  f32x2 v[AHEAD], ml[2];
  ml[0] = ask_weights(0);
  ask(v, 0, 2 * (int)threadIdx.x);
  if (p.splits > 64) ml[1] = ask_weights(64);
  T gate = (T)0.f;
  if (p.gate) gate = static_cast<const T*>(p.gate)[t * p.ldg + h];
  if (threadIdx.x < 64) {
    float m[2], l[2], top = -1e30f, sum = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bool there = (int)threadIdx.x + 64 * j < p.splits;
      m[j] = there ? ml[j][0] : -1e30f;
      l[j] = there ? ml[j][1] : 0.f;
      top = fmaxf(top, m[j]);
    }
    top = vmi_lanes::max_over<64>(top);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      m[j] = l[j] > 0.f ? exp2_hw(m[j] - top) : 0.f;   // (a part without keys holds no values)
      sum += m[j] * l[j];
    }
    sum = wave_sum(sum);
    const float g = p.gate ? sigmoid((float)gate) : 1.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) wt[threadIdx.x + 64 * j] = threadIdx.x + 64 * j < p.splits ? m[j] / sum * g : 0.f;
  }
  __syncthreads();
  if (seq < 0) return;   // (here: in front, the parts would wait for it)
  for (int k = 2 * threadIdx.x; k < p.width; k += 2 * blockDim.x) {
    f32x2 a = f32x2{0.f, 0.f};
    for (int i0 = 0; i0 < p.splits; i0 += AHEAD) {
      if (i0 > 0 || k >= 2 * (int)blockDim.x) ask(v, i0, k);
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        const float w = wt[i0 + i];
#pragma unroll
        for (int e = 0; e < 2; ++e) a[e] = fmaf(w, w != 0.f ? v[i][e] : 0.f, a[e]);   // (a part without keys holds whatever was there)
      }
    }
    T* out = static_cast<T*>(p.out) + (int64_t)t * p.ldo + (int64_t)h * p.width + k;
    typename Elem<T>::v2 o;
    o[0] = (T)a[0], o[1] = (T)a[1];
    if ((p.ldo & 1) == 0 && ((uintptr_t)p.out & (2 * sizeof(T) - 1)) == 0) *reinterpret_cast<typename Elem<T>::v2*>(out) = o;
    else out[0] = o[0], out[1] = o[1];
  }
}

template <typename T>
inline void launch_combine(const Combine& p, hipStream_t st) {
  const int threads = p.width >= 1024 ? 512 : (p.width + 127) / 128 * 64;
  auto* fn = p.splits <= 4 ? combine_kernel<T, 4> : p.splits <= 8 ? combine_kernel<T, 8> : combine_kernel<T, 16>;
  hipLaunchKernelGGL(fn, dim3((int64_t)p.T * p.heads), dim3(threads), 0, st, p);
}

}  // namespace vmi_hybrid
