// The vocabulary's product for few rows (included by gpt2_layer.hip; include/vmi_gpt2_layer.h: vmi_gpt2_head_f16): the final norm, if any, and logits.
//
// Bound by the weights' way from memory, 77 MB at GPT-2 small's sizes (4 TB/s).  us, a layer norm and the vendor's product / here, weights not in the Infinity Cache: width 768, 50257 columns,
// 1 row 21.7 / 19.5, 16 rows 22.1 / 20.7; 512, 32000, 4 rows 15.0 / 10.9; 1024, 50257, 1 row 25.9 / 24.4; without a norm level (18.1 / 18.1, 18.2 / 19.1), but the vendor's call takes
// the host 30 us, which is what the first token of a short prompt waits for.  Two row tiles were behind (32 rows 22.8 / 24.4).  One workgroup of eight waves a compute unit norms all rows into LDS once, while its first weights are
// under way; then every wave streams slabs of 16 columns of its own, 24 k-steps ahead, and no two waves meet again.  Slabs are dealt wave by wave across the
// compute units, so the last ones, fewer than there are waves, are spread over all of them.
#pragma once

namespace vmi_layer {

struct HeadParams {
  const h16* x;
  int64_t ldx;
  const int32_t* rows;   // row m is x[rows[m]] (NULL: x[m])
  const h16* gamma;      // NULL: rows as they are
  const h16* beta;
  float eps;
  const h16* w;          // tiles [ceil(N / 16)][K / 32][64 lanes][8]
  h16* y;                // [M][ldy], N columns of a row
  int64_t ldy;
  int M, N, K;
};

constexpr int HEAD_RW = 8, HEAD_CH = 12, HEAD_UNITS = 3;   // waves; k-steps of a chunk; 16-byte units of a row a lane
constexpr int HEAD_MAX_K = 64 * HEAD_UNITS * 8;
inline size_t head_lds(int K) { return (size_t)16 * (2 * K + 16); }

template <bool NORM>
__global__ __launch_bounds__(64 * HEAD_RW, 2) void head_kernel(const HeadParams p) {
  constexpr int NB = 3, CH = HEAD_CH;   // chunks of weights in registers, two of them ahead
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // rows [16][2 K + 16 bytes]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kc = lane >> 4, r16 = lane & 15;
  const int SL = (p.N + 15) >> 4, first = wave * (int)gridDim.x + (int)blockIdx.x, every = (int)gridDim.x * HEAD_RW;
  const int nks = p.K >> 5, cps = (nks + CH - 1) / CH, nch = first < SL ? ((SL - 1 - first) / every + 1) * cps : 0;
  h16x8 w[NB][CH];
  auto load = [&](h16x8(&to)[CH], int slab, int part) {   // (past a slab's last k-step: that one again, which meets nothing)
    const h16* at = p.w + ((int64_t)slab * nks * 64 + lane) * 8;
#pragma unroll
    for (int j = 0; j < CH; ++j) to[j] = *reinterpret_cast<const h16x8*>(at + (int64_t)min(part * CH + j, nks - 1) * 512);
  };
  // the chunk to ask for next, and the one at work: (slab, part); past the end the last one again
  int ls = min(first, SL - 1), lp = 0, left = nch - 1;
  auto on = [&] {
    if (left <= 0) return;
    --left;
    if (++lp == cps) lp = 0, ls += every;
  };
#pragma unroll
  for (int b = 0; b < NB - 1; ++b) load(w[b], ls, lp), on();
  const int units = p.K >> 3, ldb = 2 * p.K + 16;
  for (int m = wave; m < 16; m += HEAD_RW) {
    const int mm = min(m, p.M - 1);
    const h16* row = p.x + (int64_t)(p.rows ? p.rows[mm] : mm) * p.ldx;
    u32x4 x[HEAD_UNITS];
#pragma unroll
    for (int i = 0; i < HEAD_UNITS; ++i) x[i] = *reinterpret_cast<const u32x4*>(row + min(lane + 64 * i, units - 1) * 8);
    float rstd = 1.f, nmr = 0.f;
    if constexpr (NORM) {
      const float inv = 1.f / (float)p.K;
      float s = 0.f, q = 0.f;
#pragma unroll
      for (int i = 0; i < HEAD_UNITS; ++i)
        if (lane + 64 * i < units) {
#pragma unroll
          for (int e = 0; e < 4; ++e) ln_sum_pair(x[i][e], s);
        }
      const float neg_mean = -group_sum<64>(s) * inv;
#pragma unroll
      for (int i = 0; i < HEAD_UNITS; ++i)
        if (lane + 64 * i < units) {
#pragma unroll
          for (int e = 0; e < 4; ++e) ln_square_pair(x[i][e], neg_mean, q);
        }
      rstd = rsqrtf(group_sum<64>(q) * inv + p.eps), nmr = neg_mean * rstd;
    }
#pragma unroll
    for (int i = 0; i < HEAD_UNITS; ++i)
      if (lane + 64 * i < units) {
        const int u = (lane + 64 * i) * 8;
        u32x4 v = x[i];
        if constexpr (NORM) {
          const u32x4 g = *reinterpret_cast<const u32x4*>(p.gamma + u), b = *reinterpret_cast<const u32x4*>(p.beta + u);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = ln_pair(x[i][e], g[e], b[e], rstd, nmr);
        }
        *reinterpret_cast<u32x4*>(smem + m * ldb + u * 2) = v;
      }
  }
  __syncthreads();
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  int slab = first, part = 0;
  auto step = [&](const h16x8(&cur)[CH], h16x8(&next)[CH]) {
    load(next, ls, lp), on();
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = part * CH + j;
      if (k >= nks) break;   // (scalar)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(cur[j], *reinterpret_cast<const h16x8*>(smem + r16 * ldb + 64 * k + 16 * kc), acc, 0, 0, 0);
    }
    if (++part < cps) return;
    const int n = slab * 16 + 4 * kc;
    if (r16 < p.M) {
      h16* y = p.y + (int64_t)r16 * p.ldy + n;
      h16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (h16)acc[r];
      if (n + 4 <= p.N) {
        __builtin_memcpy(y, &o, 8);   // (rows of an odd number of columns: aligned to a half)
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < p.N) y[r] = o[r];
      }
    }
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
    part = 0, slab += every;
  };
  for (int c = 0; c < nch; c += NB) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (c + b < nch) step(w[b], w[(b + NB - 1) % NB]);
  }
}

}  // namespace vmi_layer
