// Linear layers of few rows (included by gpt2_layer.hip): a workgroup owns 16 rows and one or a few slabs of 16 columns, its waves take a part of K each,
// and everything a wave will ever read is requested before its first wait.
//
// Such a launch is a chain of latencies, so what is on the chain is counted:
//   * rows come from memory as whole lines and change into the matrix cores' layout (16 rows x 64 bytes) in LDS.  Loaded in that layout they cost
//     the address units 16 half-used lines an instruction: K 3072, 32 rows 5.9 -> 4.1 us, K 768 2.9 -> 2.4;
//   * in front of a norm half a wave owns a row, so a row's statistics meet inside the wave: mean first, then the squares around it, on registers;
//   * a workgroup takes as many slabs as it needs to leave one workgroup a compute unit: two of them share its load paths and vector units and end
//     a microsecond after one (32 rows, N 2304 behind a norm, one / two slabs: 4.2 / 3.7 us; 128 rows, N 3072, three / six: 5.7 / 5.3);
//   * all arguments are asked for at once (`need`): left to itself the compiler asks for them branch by branch, a trip to memory each (0.15 us).
// The waves' partial tiles meet in LDS; wave s adds those of slab s in the order of K and stores.
// GPT-2 small, 1 / 16 / 32 / 64 / 128 rows in a graph of such launches, before (rows in the matrix cores' layout, one slab) -> now, us:
// N 2304 behind a norm 3.6 / 3.8 / 5.0 / 5.9 / 6.8 -> 3.3 / 3.4 / 3.7 / 4.0 / 4.9, N 3072 3.9 / 4.1 / 5.3 / 6.2 / 7.3 -> 3.6 / 3.7 / 4.0 / 4.4 / 5.3,
// K 768 2.4 / 2.9 / 2.9 / 3.0 / 3.9 -> 2.2 / 2.3 / 2.4 / 2.4 / 2.7, K 3072 4.0 / 5.9 / 5.9 / 5.9 / 8.4 -> 3.7 / 4.1 / 4.1 / 4.1 / 5.1.  (An empty launch: 1.6.)
#pragma once

namespace vmi_layer {

template <class T>
__device__ __forceinline__ void need(const T& v) {
  asm volatile("" ::"s"(v));
}

// sum over 32 lanes
__device__ __forceinline__ float half_wave_sum(float v) {
  return group_sum<32>(v);
}

// where a wave's weight tiles lie: k-step t of a slab is `step` halves behind k-step 0 (packed tiles, or rows as stored)
struct WeightRows {
  const h16* at;
  int step;
  __device__ __forceinline__ WeightRows(const LinearParams& p, int slab, int nks, int lane) {
    step = p.w_packed ? 512 : 32;
    at = p.w_packed ? p.w + ((int64_t)slab * nks * 64 + lane) * 8 : p.w + (int64_t)(slab * 16 + (lane & 15)) * p.K + 8 * (lane >> 4);
  }
  __device__ __forceinline__ h16x8 load(int t) const { return *reinterpret_cast<const h16x8*>(at + (int64_t)t * step); }
};

// Partial tiles of NS slabs, one a wave, to the waves that store them: `mine` is the wave's own LDS (stride bytes a wave), no longer read
template <int RW, int NS, int EPI>
__device__ __forceinline__ void meet_and_store(const LinearParams& p, const f32x4 (&acc)[NS], unsigned char* smem, int stride, int wave, int lane, const Tail& tail,
                                               int m, int slab, bool stores) {
#pragma unroll
  for (int s = 0; s < NS; ++s) *reinterpret_cast<f32x4*>(smem + wave * stride + s * 1024 + lane * 16) = acc[s];
  __syncthreads();
  if (!stores) return;
  const int s = NS == 1 ? 0 : wave;
  f32x4 sum = *reinterpret_cast<const f32x4*>(smem + s * 1024 + lane * 16);
#pragma unroll
  for (int v = 1; v < RW; ++v) sum += *reinterpret_cast<const f32x4*>(smem + v * stride + s * 1024 + lane * 16);
  if (m < p.M) tail.store<EPI>(p, sum, m, (slab + s) * 16 + 4 * (lane >> 4), (slab + s) * 16);
}

constexpr int NORM_RW = 8;   // waves of a workgroup behind a norm: two rows each, an eighth of K each

inline size_t norm_rows_lds(int K, int ns) { return (size_t)16 * (K * 2 + 16) + (size_t)NORM_RW * ns * 1024; }

// J: at most that many k-steps a wave, and as many 16-byte units of a row a lane (32 lanes a row); NS slabs a workgroup
template <int J, int NS, int EPI>
__global__ __launch_bounds__(64 * NORM_RW, 2) void norm_rows_kernel(const LinearParams p) {
  constexpr int RW = NORM_RW;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // rows [16][2 K + 16 bytes], then the partial tiles
  need(p.x), need(p.ldx), need(p.w), need(p.bias), need(p.gamma), need(p.beta), need(p.eps), need(p.y), need(p.ldy), need(p.M), need(p.N), need(p.K), need(p.w_packed);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kc = lane >> 4, r16 = lane & 15;
  const int SL = p.N >> 4, slab = blockIdx.x * NS, m = blockIdx.y * 16 + r16;
  if (slab >= SL) return;
  const int nks = p.K >> 5, per = (nks + RW - 1) / RW, k0 = wave * per, nk = min(per, nks - k0);   // (nk <= 0: no part of K is left for it)
  // (what lies past a wave's last step, or past a row, is that last one again and meets nothing: no lane-wise condition around a load)
  auto step = [&](int j) { return min(k0 + min(j, per - 1), nks - 1); };
  const int units = nks * 4, l = lane & 31, xr = wave * 2 + (lane >> 5);
  auto unit = [&](int i) { return min(l + 32 * i, units - 1) * 8; };
  const h16* row = p.x + (int64_t)min((int)blockIdx.y * 16 + xr, p.M - 1) * p.ldx;
  u32x4 x[J], g[J], b[J];
#pragma unroll
  for (int i = 0; i < J; ++i) x[i] = *reinterpret_cast<const u32x4*>(row + unit(i));
#pragma unroll
  for (int i = 0; i < J; ++i) {
    g[i] = *reinterpret_cast<const u32x4*>(p.gamma + unit(i));
    b[i] = *reinterpret_cast<const u32x4*>(p.beta + unit(i));
  }
  h16x8 w[NS][J];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const WeightRows wr(p, min(slab + s, SL - 1), nks, lane);
#pragma unroll
    for (int j = 0; j < J; ++j) w[s][j] = wr.load(step(j));
  }
  const int ns = NS == 1 ? 0 : wave;   // the slab this wave stores
  const bool stores = wave < NS && slab + ns < SL;
  Tail tail;
  if (stores) tail.load<EPI>(p, m, (slab + ns) * 16 + 4 * kc, (slab + ns) * 16);

  const float inv = 1.f / (float)p.K;
  float s4[4] = {0.f, 0.f, 0.f, 0.f}, q4[4] = {0.f, 0.f, 0.f, 0.f};   // (four chains of dependent adds side by side)
#pragma unroll
  for (int i = 0; i < J; ++i)
    if (l + 32 * i < units) {
#pragma unroll
      for (int e = 0; e < 4; ++e) ln_sum_pair(x[i][e], s4[e]);
    }
  const float neg_mean = -half_wave_sum((s4[0] + s4[1]) + (s4[2] + s4[3])) * inv;
#pragma unroll
  for (int i = 0; i < J; ++i)
    if (l + 32 * i < units) {
#pragma unroll
      for (int e = 0; e < 4; ++e) ln_square_pair(x[i][e], neg_mean, q4[e]);
    }
  const float rstd = rsqrtf(half_wave_sum((q4[0] + q4[1]) + (q4[2] + q4[3])) * inv + p.eps), nmr = neg_mean * rstd;
  const int ldb = p.K * 2 + 16;
#pragma unroll
  for (int i = 0; i < J; ++i)
    if (l + 32 * i < units) {
      u32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ln_pair(x[i][e], g[i][e], b[i][e], rstd, nmr);
      *reinterpret_cast<u32x4*>(smem + xr * ldb + unit(i) * 2) = v;
    }
  __syncthreads();
  f32x4 acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j < nk) {   // (scalar condition)
      const h16x8 v = *reinterpret_cast<const h16x8*>(smem + r16 * ldb + 64 * (k0 + j) + 16 * kc);
#pragma unroll
      for (int s = 0; s < NS; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[s][j], v, acc[s], 0, 0, 0);
    }
  meet_and_store<RW, NS, EPI>(p, acc, smem + 16 * ldb, NS * 1024, wave, lane, tail, m, slab, stores);
}

constexpr int rows_stride(int J, int NS) { return 16 * (64 * J + 16) > NS * 1024 ? 16 * (64 * J + 16) : NS * 1024; }   // bytes of LDS a wave

// Rows that are multiplied as they are, with the residual behind: a wave brings its own part of K of the 16 rows through its own part of the LDS, no other
// wave waits for it.  RW waves, at most J k-steps each: six a wave where that is possible (K 768 over 4 / 8 waves: 2.36 / 2.51 us; K 3072 over 8 / 16: 4.38 / 4.08),
// as few more as there are past 3072 columns (a step that a wave does not have is read all the same: K 4096, N 1024 1 / 16 rows nine a wave 5.3 / 6.0, eight 4.7 / 5.1)
template <int RW, int J, int NS>
__global__ __launch_bounds__(64 * RW, RW / 4) void rows_kernel(const LinearParams p) {
  constexpr int EPI = VMI_LAYER_EPI_BIAS_RESIDUAL, LDB = 64 * J + 16, STRIDE = rows_stride(J, NS);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // [RW][STRIDE]
  need(p.x), need(p.ldx), need(p.w), need(p.bias), need(p.res), need(p.ldr), need(p.y), need(p.ldy), need(p.M), need(p.N), need(p.K), need(p.w_packed);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kc = lane >> 4, r16 = lane & 15;
  const int SL = p.N >> 4, slab = blockIdx.x * NS, m = blockIdx.y * 16 + r16;
  if (slab >= SL) return;
  const int nks = p.K >> 5, per = (nks + RW - 1) / RW, k0 = wave * per, nk = min(per, nks - k0);
  auto step = [&](int j) { return min(k0 + min(j, per - 1), nks - 1); };
  unsigned char* mine = smem + wave * STRIDE;
  u32x4 x[J];
#pragma unroll
  for (int i = 0; i < J; ++i) {   // (16 rows of 4 J units of 16 bytes; units past the row are its last one and meet nothing)
    const int u = lane + 64 * i, r = u / (4 * J), c = min(4 * k0 + u % (4 * J), 4 * nks - 1);
    x[i] = *reinterpret_cast<const u32x4*>(p.x + (int64_t)min((int)blockIdx.y * 16 + r, p.M - 1) * p.ldx + c * 8);
  }
  h16x8 w[NS][J];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const WeightRows wr(p, min(slab + s, SL - 1), nks, lane);
#pragma unroll
    for (int j = 0; j < J; ++j) w[s][j] = wr.load(step(j));
  }
  const int ns = NS == 1 ? 0 : wave;
  const bool stores = wave < NS && slab + ns < SL;
  Tail tail;
  if (stores) tail.load<EPI>(p, m, (slab + ns) * 16 + 4 * kc, (slab + ns) * 16);
#pragma unroll
  for (int i = 0; i < J; ++i) {
    const int u = lane + 64 * i;
    *reinterpret_cast<u32x4*>(mine + u / (4 * J) * LDB + u % (4 * J) * 16) = x[i];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wave's LDS accesses happen in order: only the compiler has to keep them)
  f32x4 acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j < nk) {
      const h16x8 v = *reinterpret_cast<const h16x8*>(mine + r16 * LDB + 64 * j + 16 * kc);
#pragma unroll
      for (int s = 0; s < NS; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[s][j], v, acc[s], 0, 0, 0);
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  meet_and_store<RW, NS, EPI>(p, acc, smem, STRIDE, wave, lane, tail, m, slab, stores);
}

}  // namespace vmi_layer
