// Linear layers of few rows: nothing between a wave and its operands (included by gpt2_layer.hip).
//
// linear_kernel brings a row tile into LDS, because its waves own columns and share the rows.  With few rows that is two trips through memory and
// a barrier in front of the first product.  Here a workgroup owns 16 columns of 16 rows and its EIGHT waves take an eighth of K each: a
// wave needs its part of a row once, so both operands go straight from memory to registers in the matrix cores' own layout (w: one contiguous
// KiB a k-step; x: 16 rows x 64 bytes), all of them requested before the first wait.  LayerNorm in front happens on those registers: the
// waves' parts of a row's sum and sum of squares meet in LDS, then every wave normalises what it holds.  Partial tiles meet in LDS, one
// wave adds them in order and stores.
// Bound by one trip through memory, the launch, and for K 3072 a compute unit's L1 (196 KiB at 64 bytes a clock).  GPT-2 small, 1 / 16 / 32 rows:
// N 2304 behind a norm 6.0 / 6.2 / 6.3 -> 4.2 / 4.4 / 5.6 us, N 3072 6.7 / 6.7 / 6.7 -> 4.7 / 5.0 / 6.2, N 768 4.4 / 4.6 / 5.0 -> 3.2 / 3.5 / 3.5, K 3072 7.3 -> 4.6 / 6.4 / 6.4;
// a layer's four one behind the other 25.2 / 26.2 / 26.3 -> 15.6 / 18.4 / 21.0.  (Two row tiles a workgroup, weights read once for both: 24.0 at
// 32 rows.  A row stride for K 3072 that spreads over the L2 channels: no difference.)
#pragma once

namespace vmi_layer {

constexpr int RK = 8;   // waves of a workgroup: parts of K

template <int J, bool LN, int EPI>   // at most J k-steps a wave
__global__ __launch_bounds__(64 * RK, 2) void rows_kernel(const LinearParams p) {
  __shared__ f32x4 red[RK - 1][64];
  __shared__ float sums[LN ? RK : 1][2][16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kc = lane >> 4, r16 = lane & 15;
  // (the row tiles of 16 columns go to one XCD, which then reads their weights once)
  const int RB = (p.M + 15) >> 4, SL = p.N >> 4;
  const int slab = (int)(blockIdx.x / (8 * RB)) * 8 + (int)(blockIdx.x & 7), m = (int)(blockIdx.x >> 3) % RB * 16 + r16;
  if (slab >= SL) return;
  const int nks = p.K >> 5, per = (nks + RK - 1) / RK, k0 = wave * per, nk = min(per, nks - k0);   // (nk <= 0: no part of K is left for it)

  h16x8 x[J], w[J];
  u32x4 g[LN ? J : 1], b[LN ? J : 1];
  // (steps past this wave's last read it again and meet nothing: no lane-wise condition around a load)
  auto step = [&](int j) { return min(k0 + min(j, per - 1), nks - 1); };
  const h16* row = p.x + (int64_t)min(m, p.M - 1) * p.ldx + 8 * kc;
#pragma unroll
  for (int j = 0; j < J; ++j) x[j] = *reinterpret_cast<const h16x8*>(row + 32 * step(j));
  if constexpr (LN) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      g[j] = *reinterpret_cast<const u32x4*>(p.gamma + 32 * step(j) + 8 * kc);
      b[j] = *reinterpret_cast<const u32x4*>(p.beta + 32 * step(j) + 8 * kc);
    }
  }
  const int wstep = p.w_packed ? 512 : 32;
  const h16* wp = p.w_packed ? p.w + ((int64_t)slab * nks * 64 + lane) * 8 : p.w + (int64_t)(slab * 16 + r16) * p.K + 8 * kc;
#pragma unroll
  for (int j = 0; j < J; ++j) w[j] = *reinterpret_cast<const h16x8*>(wp + (int64_t)step(j) * wstep);
  Tail tail;
  if (wave == 0) tail.load<EPI>(p, m, slab * 16 + 4 * kc, slab * 16);

  if constexpr (LN) {
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (j < nk) {   // (scalar)
        const u32x4 v = __builtin_bit_cast(u32x4, x[j]);
#pragma unroll
        for (int e = 0; e < 4; ++e) ln_stats_pair(v[e], s, q);
      }
    s = over_kc(s, [](float a, float c) { return a + c; });
    q = over_kc(q, [](float a, float c) { return a + c; });
    if (kc == 0) sums[wave][0][r16] = s, sums[wave][1][r16] = q;
    __syncthreads();
    const float inv = 1.f / (float)p.K;
    s = q = 0.f;
#pragma unroll
    for (int v = 0; v < RK; ++v) s += sums[v][0][r16], q += sums[v][1][r16];
    const float mean = s * inv, rstd = rsqrtf(fmaxf(q * inv - mean * mean, 0.f) + p.eps), nmr = -mean * rstd;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      u32x4 v = __builtin_bit_cast(u32x4, x[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ln_pair(v[e], g[j][e], b[j][e], rstd, nmr);
      x[j] = __builtin_bit_cast(h16x8, v);
    }
  }
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j < nk) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[j], x[j], acc, 0, 0, 0);
  if (wave > 0) red[wave - 1][lane] = acc;
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int v = 0; v < RK - 1; ++v) acc += red[v][lane];
  if (m < p.M) tail.store<EPI>(p, acc, m, slab * 16 + 4 * kc, slab * 16);
}

// k-steps a wave that the kernel is built for and K needs; 0: none
inline int rows_steps(int K) {
  const int per = ((K >> 5) + RK - 1) / RK;
  for (int j : {1, 2, 3, 4, 6, 8, 12, 16})
    if (per <= j) return j;
  return 0;
}

}  // namespace vmi_layer
