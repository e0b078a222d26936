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
    // This wave's part: its mean (rows times ones on the matrix cores: every lane has its own row's sum), and the squares around that, in four sums side by
    // side; then one mean of all parts, and every part's squares moved to it.  (The sum on the vector unit and a row centred anew for the affine form: 0.4 us
    // more at 32 rows.)
    h16x8 one;
#pragma unroll
    for (int e = 0; e < 8; ++e) one[e] = (h16)1.f;
    f32x4 total = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (j < nk) total = __builtin_amdgcn_mfma_f32_16x16x32_f16(one, x[j], total, 0, 0, 0);   // (scalar condition)
    const float own = nk > 0 ? total[0] * __builtin_amdgcn_rcpf((float)(32 * nk)) : 0.f;
    float d[J][8], q4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const u32x4 v = __builtin_bit_cast(u32x4, x[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) ln_centred_pair(v[e], -own, d[j][2 * e], d[j][2 * e + 1]);
      if (j < nk) {
#pragma unroll
        for (int e = 0; e < 8; ++e) q4[e & 3] = fmaf(d[j][e], d[j][e], q4[e & 3]);
      }
    }
    const float own_q = over_kc((q4[0] + q4[1]) + (q4[2] + q4[3]), [](float a, float c) { return a + c; });
    if (kc == 0) sums[wave][0][r16] = own, sums[wave][1][r16] = own_q;
    __syncthreads();
    const float inv = 1.f / (float)p.K;
    float n[RK], c[RK], s = 0.f, q = 0.f;
#pragma unroll
    for (int v = 0; v < RK; ++v) {
      n[v] = (float)(32 * max(0, min(per, nks - v * per)));   // (0: no part of K, no sums)
      c[v] = sums[v][0][r16];
      s = fmaf(n[v], c[v], s);
      q += sums[v][1][r16];
    }
    const float mean = s * inv;
#pragma unroll
    for (int v = 0; v < RK; ++v) q = fmaf(n[v] * (c[v] - mean), c[v] - mean, q);
    const float rstd = rsqrtf(q * inv + p.eps), shift = (own - mean) * rstd;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      u32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ln_affine_pair(fmaf(d[j][2 * e], rstd, shift), fmaf(d[j][2 * e + 1], rstd, shift), g[j][e], b[j][e]);
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
