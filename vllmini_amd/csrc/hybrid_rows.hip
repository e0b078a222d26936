// Products of few rows in bfloat16 (include/vmi_hybrid.h): the waves of a workgroup take a part of K each.
//
// A launch of this kind is a chain of latencies, so what is on the chip is counted: rows come from memory as whole lines and change into the matrix
// cores' layout (16 rows x 64 bytes) in LDS; all arguments are asked for at once (`need`: left to itself the compiler asks branch by branch, a trip to
// memory each); what the epilogue adds to is asked for in front of everything.  The waves' partial tiles meet in LDS; one wave a tile adds them in
// the order of K and stores.
#include "hybrid_kv_prep.hpp"
#include "hybrid_latent_prep.hpp"
#include "hybrid_linear.hpp"

namespace vmi_hybrid {

template <int EPI>
__device__ __forceinline__ void need_args(const vmi_hy_linear_args& p) {
  need(p.x), need(p.w), need(p.y), need(p.ldx), need(p.ldy), need(p.M), need(p.N), need(p.K);
  if constexpr (EPI == VMI_HY_E_STORE) need(p.bias);
  if constexpr (EPI == VMI_HY_E_GATED) need(p.gate), need(p.ldg);
  if constexpr (EPI == VMI_HY_E_GLU || EPI == VMI_HY_E_STORE_GLU) need(p.scale), need(p.glu_alpha), need(p.glu_up);
  if constexpr (EPI == VMI_HY_E_STORE_GLU) need(p.y2), need(p.ldy2), need(p.n_split);
  if constexpr (EPI == VMI_HY_E_FLOAT) need(p.scale), need(p.n_out);
}

constexpr int plain_stride(int J, int MT) { return MT * 16 * (64 * J + 16); }   // bytes of LDS a wave

// Rows as they are.  A workgroup owns 16 columns of 16 MT rows of a group; a wave brings its own part of K of the rows through its own part of the
// LDS, chunks of J k-steps, so nothing but the sum at the end waits for another wave.  NB chunks of weights in registers.  The order of the requests is the
// order of their use (they complete in order): rows of a chunk, then the weights NB - 1 chunks on.  NB = 1: a wave's part is one chunk.
// NCH > 0: NCH whole chunks a wave, K = 32 RW J NCH, all of whose requests are written out, NB chunks of rows and of weights on their way: with sizes and ends the compiler could
// not see it waited for all of them at every chunk.  XI: requests for the rows of a chunk (2 XI rows at most).  Before -> now, weights not in the Infinity Cache, us: K 6144, N 1024 1 / 16 / 32
// rows 7.9 / 9.7 / 9.4 -> 6.5 / 8.8 / 8.6, N 2048 32 rows 10.2 -> 9.4, N 4096 1 / 16 12.4 / 14.1 -> 11.1 / 13.1; K 8192, N 2048 32 rows 12.5 -> 11.4, N 4096 1 / 16 16.4 / 17.9 -> 14.5 / 16.3; K 12288,
// N 1024 12.0 / 16.0 -> 11.0 / 14.7, N 4096 21.9 / 23.8 -> 20.3 / 22.6 (101 MB, 5.0 TB/s).
// XK = VMI_HY_X_CONCAT: rows of x and x2 side by side, float32, rounded on their way into LDS (half of K is whole units, and of whole chunks a wave's part lies in one).
template <int RW, int J, int MT, int NB, int EPI, int NCH = 0, int XI = J, int XK = VMI_HY_X_ROWS>
__device__ __forceinline__ void plain_rows_slab(const vmi_hy_linear_args& p, const int slab, const int m0, const int grp, unsigned char* const smem) {
  constexpr bool CAT = XK == VMI_HY_X_CONCAT;
  using XT = std::conditional_t<CAT, float, b16>;
  auto rounded = [](const V8<XT>& v) {
    if constexpr (CAT) return from_f32<b16>(v);
    else return v;
  };
  constexpr int LDB = 64 * J + 16, STRIDE = plain_stride(J, MT);
  need_args<EPI>(p), need(p.x_gstride), need(p.y_gstride);
  if constexpr (CAT) need(p.x2);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kc = lane >> 4, r16 = lane & 15;
  if (slab * 16 >= p.N) return;
  const int nks = p.K >> 5, per = (nks + RW - 1) / RW, k0 = wave * per, nk = min(per, nks - k0);   // (nk <= 0: no part of K is left for it)
  const int nch = (per + J - 1) / J, rows = p.M - m0;
  const int m = m0 + (MT == 1 ? 0 : wave * 16) + r16, n = slab * 16 + 4 * kc;   // (what this wave stores, if it does)
  const bool stores = wave < MT && m < p.M;
  [[maybe_unused]] f32x4 before = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (EPI == VMI_HY_E_RESIDUAL)
    if (stores) before = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.y) + (int64_t)m * p.ldy + (int64_t)grp * p.y_gstride + n);

  const XT* xp = static_cast<const XT*>(p.x) + (int64_t)grp * p.x_gstride;
  [[maybe_unused]] const XT* x2p = CAT ? static_cast<const XT*>(p.x2) - (p.K >> 1) : nullptr;   // (column c of the second half: x2p[c])
  const b16* wp = static_cast<const b16*>(p.w) + (((int64_t)grp * (p.N >> 4) + slab) * nks * 64 + lane) * 8;
  unsigned char* mine = smem + wave * STRIDE;
  f32x4 acc[MT];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) acc[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (NCH > 0) {
    static_assert(MT == 1, "one row tile");
    V8<XT> xc[NB][XI];
    b16x8 wc[NB][J];
    const int u0 = 4 * k0 + lane % (4 * J), r0 = lane / (4 * J);   // (request i of a chunk: rows r0 + 2 i)
    static_assert(4 * J == 32, "two rows a request");
    const XT* xr[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) xr[i] = (CAT && wave >= RW / 2 ? x2p : xp) + (int64_t)min(m0 + r0 + 2 * i, p.M - 1) * p.ldx + u0 * 8;
    const b16* wr = wp + (int64_t)k0 * 512;
    auto ask = [&](int b, int c) {   // (in the order of their use, which is the order they come in)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < XI; ++i) xc[b][i] = load8(xr[i] + c * (32 * J));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < J; ++j) wc[b][j] = load8(wr + (c * J + j) * 512);
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int b = 0; b < NB; ++b) ask(b, b);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
#pragma unroll
      for (int i = 0; i < XI; ++i) *reinterpret_cast<b16x8*>(mine + (r0 + 2 * i) * LDB + lane % (4 * J) * 16) = rounded(xc[c % NB][i]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wave's LDS accesses happen in order: only the compiler has to keep them)
#pragma unroll
      for (int j = 0; j < J; ++j) mma(acc[0], wc[c % NB][j], *reinterpret_cast<const b16x8*>(mine + r16 * LDB + 64 * j + 16 * kc));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (c + NB < NCH) ask(c % NB, c + NB);
    }
  } else {
    V8<XT> x[MT][J];
    b16x8 w[NB][J];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
      for (int i = 0; i < J; ++i) x[mi][i] = zero8<XT>();
    // (16 rows of 4 J units of 16 bytes; units past the row are its last one and meet nothing; 64 units that lie past M altogether stay away)
    auto load_x = [&](int c) {
#pragma unroll
      for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int i = 0; i < J; ++i)
          if (mi * 16 + 64 * i / (4 * J) < rows) {   // (scalar)
            const int u = lane + 64 * i, r = u / (4 * J), col = min(4 * (k0 + c * J) + u % (4 * J), 4 * nks - 1);
            x[mi][i] = load8((CAT && 16 * col >= p.K ? x2p : xp) + (int64_t)min(m0 + mi * 16 + r, p.M - 1) * p.ldx + col * 8);
          }
    };
    auto load_w = [&](b16x8(&dst)[J], int c) {
#pragma unroll
      for (int j = 0; j < J; ++j) dst[j] = load8(wp + (int64_t)min(k0 + min(c * J + j, per - 1), nks - 1) * 512);
    };
    load_x(0);
#pragma unroll
    for (int b = 0; b < (NB > 1 ? NB - 1 : 1); ++b) load_w(w[b], b);
    auto chunk = [&](int c, b16x8(&cur)[J], b16x8(&last)[J]) {
#pragma unroll
      for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int i = 0; i < J; ++i) {
          const int u = lane + 64 * i;
          *reinterpret_cast<b16x8*>(mine + (mi * 16 + u / (4 * J)) * LDB + u % (4 * J) * 16) = rounded(x[mi][i]);
        }
      if constexpr (NB > 1) {
        if (c + 1 < nch) load_x(c + 1);
        load_w(last, c + NB - 1);   // (past the end: a tile again, a cache hit)
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wave's LDS accesses happen in order: only the compiler has to keep them)
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (c * J + j < nk) {   // (scalar)
#pragma unroll
          for (int mi = 0; mi < MT; ++mi) mma(acc[mi], cur[j], *reinterpret_cast<const b16x8*>(mine + (mi * 16 + r16) * LDB + 64 * j + 16 * kc));
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    for (int c = 0; c < nch; c += NB) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (c + b < nch) chunk(c + b, w[b], w[(b + NB - 1) % NB]);
    }
  }
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) *reinterpret_cast<f32x4*>(mine + mi * 1024 + lane * 16) = acc[mi];
  __syncthreads();
  if (!stores) return;
  const unsigned char* at = smem + (MT == 1 ? 0 : wave) * 1024 + lane * 16;
  f32x4 sum = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
  for (int v = 1; v < RW; ++v) sum += *reinterpret_cast<const f32x4*>(at + v * STRIDE);
  if constexpr (EPI == VMI_HY_E_RESIDUAL)
    *reinterpret_cast<f32x4*>(static_cast<float*>(p.y) + (int64_t)m * p.ldy + (int64_t)grp * p.y_gstride + n) = before + sum;
  else
    epilogue<b16, EPI>(p, sum, m, n, slab * 16, grp);
}
template <int RW, int J, int MT, int NB, int EPI, int NCH = 0, int XI = J, int XK = VMI_HY_X_ROWS>
__global__ __launch_bounds__(64 * RW, RW / 4) void plain_rows_kernel(const vmi_hy_linear_args p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // [RW][plain_stride]
  plain_rows_slab<RW, J, MT, NB, EPI, NCH, XI, XK>(p, blockIdx.x, blockIdx.y * 16 * MT, blockIdx.z, smem);
}

// A product by heads and what a token's attention needs besides: two launches of a chain that do not read each other's results, in one.  The
// first T workgroups take a token each, the others a slab of 16 columns of 16 MT rows of a head.  Few rows, each is little more than its launch: queries into the latent space beside
// latent_prep, 8 heads of 128 into 512, 12 rows, us: 4.2 + 4.9 -> 4.8; width 1024, 12 sequences, 24 tokens 7311 -> 7203 (of one sequence, width 4096, less than two runs of it differ by).
// The gates' products (2 of 2048 x 128, 32 rows) beside kv_prep 4.5 + 5.1 -> 5.0.
struct LatentPrep {
  vmi_hy_latent_prep_args a;
  __device__ __forceinline__ void token(const vmi_hy_step& s, int t, unsigned char* smem) const { latent_prep_token<b16, false>(a, s, nullptr, t, reinterpret_cast<float*>(smem)); }
};
struct LatentPromptPrep {
  vmi_hy_latent_prep_args a;
  b16* rows;
  int row0;
  bool mixed;
  __device__ __forceinline__ void token(const vmi_hy_step& s, int t, unsigned char* smem) const {
    latent_prompt_prep_token(a, s, rows, row0, mixed, t, reinterpret_cast<float*>(smem));
  }
};
struct KvPrep {
  vmi_hy_kv_prep_args a;
  __device__ __forceinline__ void token(const vmi_hy_step& s, int t, unsigned char*) const { kv_prep_token<b16>(a, s, t); }
};
template <int J, int MT, class Prep>
__global__ __launch_bounds__(256, 1) void rows_beside_kernel(const vmi_hy_linear_args p, const Prep prep, const vmi_hy_step s, const int slabs, const int blocks) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int at = (int)blockIdx.x - s.T;
  if (at < 0) {
    prep.token(s, blockIdx.x, smem);
  } else {
    const int rest = at / slabs, grp = rest / blocks;
    plain_rows_slab<4, J, MT, 1, VMI_HY_E_STORE>(p, at - rest * slabs, (rest - grp * blocks) * 16 * MT, grp, smem);
  }
}

// Rows of the element type over many columns, 16 MT of them: eight waves hold an eighth of K of all rows each, in registers and in the matrix cores' layout,
// and the workgroup walks over slabs of 16 columns, blockIdx, blockIdx + grid, ..; the ring of weight tiles runs on across slabs.  NCH chunks of 4 k-steps are a
// wave's part of a slab, NB chunks are in registers.  A slab's partial tiles meet in LDS (two places, one barrier a slab); another wave each time adds a
// tile's in the order of K and stores.  Nothing in the walk depends on a condition but its end and the stores: the compiler counts loads
// in flight, and where paths meet that differ in them it waits for all.  With sizes and ends it could not see, the ring ran empty every three slabs.  Norm and
// product, us, before -> without conditions: K 2048, N 12288 9 / 32 / 47 rows 15.5 / 18.0 / 19.0 -> 14.2 / 16.7 / 17.2, N 20480 20.8 / 23.2 / 25.6 -> 19.4 / 22.3 / 24.1, N 6144 32
// rows 13.9 -> 12.5; K 3072, N 6144 47 rows 17.6 -> 15.6; K 1024, N 24576 18.5 -> 16.7.  (84 MB alone, nothing computed: 15.2.)
constexpr size_t HELD_LDS = 2 * 8 * 1024;   // ... a row tile

template <int NCH, int MT, int NB, int EPI>
__global__ __launch_bounds__(512, 2) void held_rows_kernel(const vmi_hy_linear_args p, const int slabs) {
  constexpr int W = 8, CS = 4, KS = NCH * CS, NKS = W * KS;   // k-steps of a wave, of a slab: K = 1024 NCH
  static_assert(NB % NCH == 0, "a chunk's place in its slab follows from its place in the ring");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // [2][W][MT][1024]
  need_args<EPI>(p), need(slabs);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kc = lane >> 4, r16 = lane & 15;
  const int m0 = blockIdx.y * 16 * MT, k0 = wave * KS;
  if ((int)blockIdx.x >= slabs) return;
  b16x8 x[KS][MT], wb[NB][CS];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) {
    const b16* row = static_cast<const b16*>(p.x) + (int64_t)min(m0 + mi * 16 + r16, p.M - 1) * p.ldx + 8 * kc + 32 * k0;
#pragma unroll
    for (int j = 0; j < KS; ++j) x[j][mi] = load8(row + 32 * j);
  }
  __builtin_amdgcn_sched_barrier(0);   // (requests in the order of their use, also where the compiler would turn them round: they complete in order)
  int ls = blockIdx.x;   // the slab to load from next
  auto load_w = [&](b16x8(&dst)[CS], int c) {
    // (past the last slab: 16 bytes of it for all lanes, which meet nothing; a condition around a load makes every wait a wait for all)
    const bool past = ls >= slabs;
    const b16* at = static_cast<const b16*>(p.w) + ((int64_t)(past ? (int)blockIdx.x : ls) * NKS + k0 + c * CS) * 512 + (past ? 0 : lane * 8);
#pragma unroll
    for (int j = 0; j < CS; ++j) dst[j] = load8(at + j * 512);
    __builtin_amdgcn_sched_barrier(0);
    if (c == NCH - 1) ls += gridDim.x;
  };
#pragma unroll
  for (int b = 0; b < NB - 1; ++b) load_w(wb[b], b % NCH);
  int i = 0, slab = blockIdx.x;
  // a slab whose first chunk is in place B0 of the ring; more: its chunks' successors are asked for
  auto walk = [&](auto b0, bool more) {
    constexpr int B0 = decltype(b0)::value;
    f32x4 acc[MT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) acc[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      if (more) load_w(wb[(B0 + c + NB - 1) % NB], (c + NB - 1) % NCH);
#pragma unroll
      for (int j = 0; j < CS; ++j)
#pragma unroll
        for (int mi = 0; mi < MT; ++mi) mma(acc[mi], wb[B0 + c][j], x[c * CS + j][mi]);
    }
    unsigned char* to = smem + (i & 1) * W * MT * 1024;
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) *reinterpret_cast<f32x4*>(to + (wave * MT + mi) * 1024 + lane * 16) = acc[mi];
    __syncthreads();   // (two places: who still adds up slab i has not passed the barrier of slab i + 1)
    const int mi = (wave - i * MT) & (W - 1);
    if (mi < MT) {
      f32x4 sum = *reinterpret_cast<const f32x4*>(to + mi * 1024 + lane * 16);
#pragma unroll
      for (int v = 1; v < W; ++v) sum += *reinterpret_cast<const f32x4*>(to + (v * MT + mi) * 1024 + lane * 16);
      const int m = m0 + mi * 16 + r16;
      if (m < p.M) epilogue<b16, EPI>(p, sum, m, slab * 16 + 4 * kc, slab * 16, 0);
    }
    ++i;
    slab += gridDim.x;
  };
  // Whole rounds of the ring, then what is left, which the ring holds.  One way out of the loop: any other joins the way back in the compiler's eyes
  // (a return as well), and then the places of the ring are in an unknown order and a third of the waits are waits for all.
  constexpr int ROUND = NB / NCH;
  static_assert((ROUND <= 3 || ROUND == 6) && (ROUND - 1) * NCH <= NB - 1, "the slabs behind the last round are in the ring");
  for (; slab + (ROUND - 1) * (int)gridDim.x < slabs;) {
    walk(std::integral_constant<int, 0>{}, true);
    if constexpr (ROUND > 1) walk(std::integral_constant<int, NCH % NB>{}, true);
    if constexpr (ROUND > 2) walk(std::integral_constant<int, 2 * NCH % NB>{}, true);
    if constexpr (ROUND > 3) walk(std::integral_constant<int, 3 * NCH % NB>{}, true);
    if constexpr (ROUND > 4) walk(std::integral_constant<int, 4 * NCH % NB>{}, true);
    if constexpr (ROUND > 5) walk(std::integral_constant<int, 5 * NCH % NB>{}, true);
  }
  if constexpr (ROUND > 1) {
    if (slab >= slabs) return;
    walk(std::integral_constant<int, 0>{}, false);
  }
  if constexpr (ROUND > 2) {
    if (slab >= slabs) return;
    walk(std::integral_constant<int, NCH % NB>{}, false);
  }
  if constexpr (ROUND > 3) {
    if (slab >= slabs) return;
    walk(std::integral_constant<int, 2 * NCH % NB>{}, false);
    if (slab >= slabs) return;
    walk(std::integral_constant<int, 3 * NCH % NB>{}, false);
    if (slab >= slabs) return;
    walk(std::integral_constant<int, 4 * NCH % NB>{}, false);
  }
}

inline size_t norm_rows_lds(int K, int rw, int ns) { return (size_t)16 * (K * 2 + 16) + (size_t)rw * ns * 1024; }

// Rows behind a norm (float32).  Half a wave owns a row, so its statistics meet inside the wave: mean first, then the squares around it, on registers.  A
// workgroup takes NS slabs of 16 columns, as many as leave one workgroup a compute unit: two of them share its load paths and vector units.
// J: at most that many k-steps a wave, and half as many 16-byte units of a row a lane.
template <int RW, int J, int NS, bool FULL, int EPI>
__global__ __launch_bounds__(64 * RW, RW / 4) void norm_rows_kernel(const vmi_hy_linear_args p) {
  constexpr int LPR = 4 * RW, U = 2 * J;   // lanes a row, 16-byte units of a row a lane
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // rows [16][2 K + 16 bytes], then the partial tiles [RW][NS][1024]
  need_args<EPI>(p), need(p.rows), need(p.norm_w), need(p.norm_n), need(p.rms), need(p.eps);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kc = lane >> 4, r16 = lane & 15;
  const int SL = p.N >> 4, slab = blockIdx.x * NS, m = blockIdx.y * 16 + r16;
  if (slab >= SL) return;
  const int nks = FULL ? RW * J : p.K >> 5, per = FULL ? J : (nks + RW - 1) / RW, k0 = wave * per, nk = FULL ? J : min(per, nks - k0);
  auto step = [&](int j) { return FULL ? k0 + j : min(k0 + min(j, per - 1), nks - 1); };
  auto row_sum = [](float v) { return vmi_lanes::sum_over<LPR>(v); };
  const int units = nks * 8, l = lane % LPR, xr = (wave * 64 + lane) / LPR, mm = min((int)blockIdx.y * 16 + xr, p.M - 1);
  // (what lies past a row, or past a wave's last k-step, is that last one again and meets nothing: no lane-wise condition around a load)
  auto unit = [&](int i) { return (FULL ? l + LPR * i : min(l + LPR * i, units - 1)) * 4; };
  const float* row = static_cast<const float*>(p.x) + (int64_t)(p.rows ? p.rows[mm] : mm) * p.ldx;
  f32x4 x[U], g[U];
#pragma unroll
  for (int i = 0; i < U; ++i) x[i] = *reinterpret_cast<const f32x4*>(row + unit(i));
#pragma unroll
  for (int i = 0; i < U; ++i) g[i] = *reinterpret_cast<const f32x4*>(p.norm_w + unit(i));
  b16x8 w[NS][J];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const b16* wp = static_cast<const b16*>(p.w) + ((int64_t)min(slab + s, SL - 1) * nks * 64 + lane) * 8;
#pragma unroll
    for (int j = 0; j < J; ++j) w[s][j] = load8(wp + (int64_t)step(j) * 512);
  }
  // (only the first norm_n columns are normed: what lies behind them may be anything, and comes out as zeros)
  auto clear_behind = [&]() {
    if (p.norm_n < p.K) {   // (scalar)
#pragma unroll
      for (int i = 0; i < U; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[i][e] = (l + LPR * i) * 4 + e < p.norm_n ? x[i][e] : 0.f;
    }
  };
  auto there = [&](int i) { return FULL || l + LPR * i < units; };
  const float inv = 1.f / (float)p.norm_n;
  clear_behind();
  if (!p.rms) {
    float s4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (there(i)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s4[e] += x[i][e];
      }
    const float mean = row_sum((s4[0] + s4[1]) + (s4[2] + s4[3])) * inv;
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[i][e] -= mean;
    clear_behind();
  }
  float q4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < U; ++i)
    if (there(i)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) q4[e] = fmaf(x[i][e], x[i][e], q4[e]);
    }
  const float rstd = 1.f / sqrtf(row_sum((q4[0] + q4[1]) + (q4[2] + q4[3])) * inv + p.eps);
  const int ldb = (FULL ? 64 * RW * J : p.K * 2) + 16;
#pragma unroll
  for (int i = 0; i < U; ++i)
    if (there(i)) {
      b16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (b16)(x[i][e] * rstd * g[i][e]);
      *reinterpret_cast<b16x4*>(smem + xr * ldb + unit(i) * 2) = v;
    }
  __syncthreads();
  f32x4 acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j < nk) {   // (scalar)
      const b16x8 v = *reinterpret_cast<const b16x8*>(smem + r16 * ldb + 64 * (k0 + j) + 16 * kc);
#pragma unroll
      for (int s = 0; s < NS; ++s) mma(acc[s], w[s][j], v);
    }
  unsigned char* parts = smem + 16 * ldb;
#pragma unroll
  for (int s = 0; s < NS; ++s) *reinterpret_cast<f32x4*>(parts + (wave * NS + s) * 1024 + lane * 16) = acc[s];
  __syncthreads();
  const int s = NS == 1 ? 0 : wave;   // the slab this wave stores
  if (wave >= NS || slab + s >= SL || m >= p.M) return;
  f32x4 sum = *reinterpret_cast<const f32x4*>(parts + s * 1024 + lane * 16);
#pragma unroll
  for (int v = 1; v < RW; ++v) sum += *reinterpret_cast<const f32x4*>(parts + (v * NS + s) * 1024 + lane * 16);
  epilogue<b16, EPI>(p, sum, m, (slab + s) * 16 + 4 * kc, (slab + s) * 16, 0);
}

// out[t] = the norm of x[rows[t]] in the element type, a workgroup a row; everything asked for at once, U 16-byte units a thread (K <= 2048 U).  Few rows stand
// between two products here, and what counts is how soon the second one starts: 4.1 us of a chain of launches with a row's weight asked for behind its statistics, 2.8 so
template <int U>
__global__ __launch_bounds__(512) void norm_few_kernel(const vmi_hy_linear_args p) {
  need(p.x), need(p.ldx), need(p.rows), need(p.norm_w), need(p.normed), need(p.norm_n), need(p.K), need(p.eps), need(p.rms);
  __shared__ float part[2][8];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* row = static_cast<const float*>(p.x) + (int64_t)(p.rows ? p.rows[t] : t) * p.ldx;
  f32x4 v[U], w[U];
#pragma unroll
  for (int i = 0; i < U; ++i) v[i] = *reinterpret_cast<const f32x4*>(row + min((tid + i * 512) * 4, p.K - 4));
#pragma unroll
  for (int i = 0; i < U; ++i) w[i] = *reinterpret_cast<const f32x4*>(p.norm_w + min((tid + i * 512) * 4, p.K - 4));
  auto clear_behind = [&]() {   // (the columns that are normed: what lies behind them may be anything)
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = (tid + i * 512) * 4 + e < p.norm_n ? v[i][e] : 0.f;
  };
  auto all = [&](float s, float(&at)[8]) {
    s = wave_sum(s);
    if (lane == 0) at[wave] = s;
    __syncthreads();
    return ((at[0] + at[1]) + (at[2] + at[3])) + ((at[4] + at[5]) + (at[6] + at[7]));
  };
  const float inv = 1.f / (float)p.norm_n;
  clear_behind();
  if (!p.rms) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < U; ++i) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
    const float mean = all(s, part[0]) * inv;
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] -= mean;
    clear_behind();
  }
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < U; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) q = fmaf(v[i][e], v[i][e], q);
  const float rstd = 1.f / sqrtf(all(q, part[1]) * inv + p.eps);
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const int k = (tid + i * 512) * 4;
    b16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (b16)(v[i][e] * rstd * w[i][e]);
    if (k < p.K) *reinterpret_cast<b16x4*>(static_cast<b16*>(p.normed) + (int64_t)t * p.K + k) = o;
  }
}

// ---- which, and how -------------------------------------------------------------------------------------------------------------

template <typename F>
static int launch(F* fn, const vmi_hy_linear_args& p, dim3 grid, int threads, size_t lds, hipStream_t st) {
  if (int rc = allow_lds(fn, lds, "vmi_hy_linear")) return rc;
  hipLaunchKernelGGL(fn, grid, dim3(threads), lds, st, p);
  return launched("vmi_hy_linear");
}
// (a multiple of 8 column blocks: the row tiles of one then go to one XCD, which reads their weights once)
static unsigned blocks8(int n) { return (unsigned)(n + 7) / 8 * 8; }

int launch_norm_few(const vmi_hy_linear_args& p, hipStream_t st) {
  switch ((p.K + 2047) / 2048) {
    case 1: return launch(norm_few_kernel<1>, p, dim3(p.M), 512, 0, st);
    case 2: return launch(norm_few_kernel<2>, p, dim3(p.M), 512, 0, st);
    case 3:
    case 4: return launch(norm_few_kernel<4>, p, dim3(p.M), 512, 0, st);
    default: return -1;   // (longer rows: add_norm_kernel)
  }
}

// Slabs a workgroup of norm_rows_kernel takes: as few as leave one workgroup a compute unit; 0: the kernel is not built for these sizes, or they are more than
// that.  Rows of up to 2048 columns; past 1024 sixteen waves share one, whose registers hold two slabs.
int norm_slabs(int M, int N, int K) {
  const int nks = K >> 5, rb = (M + 15) >> 4;
  if (nks > 64) return 0;
  for (int ns : {1, 2, 3, 4, 6}) {
    if (ns > 2 && nks > 32) break;
    if ((ns == 3 || ns == 6) && nks != 32) continue;
    if ((int64_t)(((N >> 4) + ns - 1) / ns) * rb <= 256) return ns;
  }
  return 0;
}
// rows_kernel's forerunner (an eighth of K a wave, rows in the matrix cores' layout), resident_kernel or linear_kernel, whichever was ahead / norm_rows_kernel, in a graph of such
// launches, us: K 1024, N 2048 1 / 12 / 32 / 40 rows 4.7 / 5.6 / 6.0 / 8.6 -> 4.2 / 4.4 / 4.5 / 4.8, N 6144 6.5 / 8.2 / 11.2 / 18.5 -> 5.2 / 5.3 / 5.6 / 6.5, N 10240 8.1 / 9.9 / 13.8
// (32) -> 6.4 / 6.3 / 7.1; K 2048, N 4096 7.7 / 9.8 / 15.3 (32) -> 7.1 / 7.5 / 8.5.  Of widths in between (K 1152 to 1920, the forerunner's sizes), 1 / 12 / 32 / 47 rows: K 1152, N 2048 6.1 / 7.9 / 8.5 / 14.2 -> 5.6 / 5.7 / 5.8 /
// 6.6; K 1280, N 4096 6.5 / 8.1 / 10.5 (32) -> 5.9 / 5.9 / 6.8; K 1792, N 512 6.2 / 8.1 / 8.7 / 8.7 -> 5.5 / 5.7 / 5.9 / 5.9; K 1920, N 4096 7.4 / 9.1 / 12.7 (32) -> 6.4 / 6.5 / 7.5.  More than a workgroup a compute unit: K 1024, N 10240, 40 rows 11.5 here, 11.0 in held_rows_kernel.

template <int RW, int J, bool FULL, int EPI>
static int norm_rows_of(const vmi_hy_linear_args& p, int ns, hipStream_t st) {
  auto go = [&](auto* fn) { return launch(fn, p, dim3(blocks8(((p.N >> 4) + ns - 1) / ns), (p.M + 15) >> 4), 64 * RW, norm_rows_lds(p.K, RW, ns), st); };
  if (ns == 1) return go(norm_rows_kernel<RW, J, 1, FULL, EPI>);
  if (ns == 2) return go(norm_rows_kernel<RW, J, 2, FULL, EPI>);
  if constexpr (RW == 8) {
    if (ns == 4) return go(norm_rows_kernel<RW, J, 4, FULL, EPI>);
    if constexpr (J == 4 && FULL) {
      if (ns == 3) return go(norm_rows_kernel<RW, J, 3, FULL, EPI>);
      if (ns == 6) return go(norm_rows_kernel<RW, J, 6, FULL, EPI>);
    }
  }
  return fail(VMI_HY_E_ARG, "vmi_hy_linear", "not built");   // (norm_slabs names no other)
}

template <int EPI>
static int norm_rows_epi(const vmi_hy_linear_args& p, hipStream_t st) {
  const int nks = p.K >> 5, ns = norm_slabs(p.M, p.N, p.K);
  if (nks == 64) return norm_rows_of<16, 4, true, EPI>(p, ns, st);
  if (nks == 48) return norm_rows_of<16, 3, true, EPI>(p, ns, st);
  if (nks == 32) return norm_rows_of<8, 4, true, EPI>(p, ns, st);
  if (nks == 24) return norm_rows_of<8, 3, true, EPI>(p, ns, st);
  if (nks == 16) return norm_rows_of<8, 2, true, EPI>(p, ns, st);
  if (nks == 8) return norm_rows_of<8, 1, true, EPI>(p, ns, st);
  if (nks > 32) return norm_rows_of<16, 4, false, EPI>(p, ns, st);
  return nks <= 16 ? norm_rows_of<8, 2, false, EPI>(p, ns, st) : norm_rows_of<8, 4, false, EPI>(p, ns, st);
}

int launch_norm_rows(const vmi_hy_linear_args& p, hipStream_t st) {
  switch (p.epilogue) {
    case VMI_HY_E_STORE: return norm_rows_epi<VMI_HY_E_STORE>(p, st);
    case VMI_HY_E_FLOAT: return norm_rows_epi<VMI_HY_E_FLOAT>(p, st);
    case VMI_HY_E_GLU: return norm_rows_epi<VMI_HY_E_GLU>(p, st);
    default: return norm_rows_epi<VMI_HY_E_STORE_GLU>(p, st);
  }
}

// Whether rows that have been normed by a launch of their own go to held_rows_kernel: 9 to 64 of them, whose waves' parts of K are whole chunks, K % 1024 == 0 (a condition around a
// chunk's products costs the ring), up to the 4096 that registers hold.
//
// Below 4096 columns rows are normed for it, where norm_rows_kernel does not take them and resident_kernel, whose workgroups would norm all each, is behind or takes
// no more than 32.  At 4096 norm_first norms them anyway, and a workgroup walks a slab of that length alone: with few slabs the waves of plain_rows_kernel (or
// linear_kernel, with what it stores gated) end sooner.
//
// Both launches, us, weights not in the Infinity Cache, the other kernels / this one (the walk before it lost its conditions, without which K 1024 to 3072 end 3 to 10 per cent sooner):
//   K 1024  N 50272  40 rows 49.5 / 22.1
//   K 2048  N 12288   8 14.9 / 14.9   12 17.8 / 15.0   32 21.6 / 17.3   40 41.8 / 17.2
//           N 20480   8 19.0 / 19.9   12 22.3 / 19.9   32 26.8 / 22.2   40 47.8 / 23.5
//           N 50272   8 39.4 / 41.3   12 42.3 / 41.6   32 50.4 / 45.7   40 95.1 / 48.8
//   K 3072  N   512  33 26.2 / 12.6   47 27.2 / 12.6   64 31.7 / 13.7       (9 to 32 rows stay with resident_kernel,
//           N  4096  33 27.9 / 14.3   47 28.8 / 14.7   64 33.4 / 16.4        which is behind too from N 2048 on:
//           N 24576  33 57.5 / 35.2   47 57.0 / 37.2   64 58.2 / 39.0        N 6144, 16 rows 17.7, 14.3 here)
//   K 4096  16 / 24 / 32 rows: N 4096 12.3 / 13.3, 13.9 / 17.6, 17.9 / 16.5 (40 rows gated 27.5 / 16.9)     N 6144 17.9 / 16.2, 21.1 / 20.2, 27.7 / 20.0 (32, weights in that cache, 15.5 / 18.5)
//           N 8192 19.0 / 19.1, 22.5 / 23.1, 28.7 / 23.0     N 12288 26.6 / 23.7, 30.4 / 28.4, 32.8 / 28.8     N 50272 85.3 / 85.5, 97.0 / 83.2, 108 / 87.7
bool held_rows_pay(int M, int N, int K, bool stored) {
  if (M < 9 || M > 64 || norm_slabs(M, N, K) > 0) return false;
  if (K == 4096) return M <= 16 ? N >= 6144 : M <= 32 ? N >= 12288 : N >= 4096 || !stored;
  return K == 2048 || ((K == 1024 || K == 3072) && M > 32);
}

template <int NCH, int MT, int NB, int EPI>
static int held_rows_of(const vmi_hy_linear_args& p, hipStream_t st) {
  auto* fn = held_rows_kernel<NCH, MT, NB, EPI>;
  const int slabs = p.N >> 4, rb = (p.M + 16 * MT - 1) / (16 * MT), most = 256 / rb / 8 * 8;   // (one workgroup a compute unit in all)
  if (int rc = allow_lds(fn, HELD_LDS * MT, "vmi_hy_linear")) return rc;
  hipLaunchKernelGGL(fn, dim3(slabs < most ? blocks8(slabs) : most, rb), dim3(512), HELD_LDS * MT, st, p, slabs);
  return launched("vmi_hy_linear");
}

template <int EPI>
static int held_rows_epi(const vmi_hy_linear_args& p, hipStream_t st) {
  switch (p.K * 4 + (p.M > 16 ? 2 : 1)) {
    case 1024 * 4 + 2: return held_rows_of<1, 2, 6, EPI>(p, st);
    case 2048 * 4 + 1: return held_rows_of<2, 1, 6, EPI>(p, st);
    case 2048 * 4 + 2: return held_rows_of<2, 2, 6, EPI>(p, st);
    case 3072 * 4 + 2: return held_rows_of<3, 2, 6, EPI>(p, st);
    case 4096 * 4 + 1: return held_rows_of<4, 1, 4, EPI>(p, st);
    case 4096 * 4 + 2: return held_rows_of<4, 2, 4, EPI>(p, st);
    default: return fail(VMI_HY_E_ARG, "vmi_hy_linear", "not built");   // (held_rows_pay names no other)
  }
}

int launch_held_rows(const vmi_hy_linear_args& p, hipStream_t st) {
  switch (p.epilogue) {
    case VMI_HY_E_STORE: return held_rows_epi<VMI_HY_E_STORE>(p, st);
    case VMI_HY_E_FLOAT: return held_rows_epi<VMI_HY_E_FLOAT>(p, st);
    case VMI_HY_E_GLU: return held_rows_epi<VMI_HY_E_GLU>(p, st);
    default: return held_rows_epi<VMI_HY_E_STORE_GLU>(p, st);
  }
}

// Rows as they are go to plain_rows_kernel where it is ahead of linear_kernel; past 64 rows there are tiles.  In a graph of such launches, us, linear_kernel / here:
//   K  1024  N 1024   1 row 3.7 / 2.9     16 4.0 / 3.1     32 4.1 / 3.1     64 6.4 / 3.2
//   K  3072  N 1024   1  4.8 / 3.8     16 5.4 / 4.4     32 5.5 / 4.5     64 13.0 / 4.6
//   K  4096  N 4096   1 10.1 / 8.1     16 11.3 / 9.0    32 12.4 / 10.7   64 24.6 / 17.1
//   8 groups of K 128, N 512  1 3.7 / 2.3   16 3.9 / 2.4   32 4.0 / 2.5   64 3.4 / 2.6      of K 512, N 128  1 4.0 / 2.5   16 4.5 / 2.7   32 4.5 / 2.7   64 5.1 / 2.7
//
// Every workgroup brings the rows again, so past one slab a compute unit (256) it is ahead only while the rows are few or short:
//   K  2048  N 16384  1 13.6 / 12.7    32 13.8 / 16.8   64 16.2 / 30.8      N 50272 1 42.8 / 35.0
//   K  4096  N  8192  8 14.2 / 13.7    24 14.0 / 15.2   64 20.7 / 28.5      N 16384 16 22.9 / 24.8
//   K   512  N 16384 32  7.1 / 6.1     N 8192 64 5.5 / 6.0                  K 128  N 50272 32 10.5 / 7.7
//   groups of K 128, N 512, 47 rows: 32 of them 4.2 / 4.1, 64 5.3 / 5.9; N 576 (linear_kernel's nine column blocks of a group padded to sixteen) 5.0 / 4.4, 8.0 / 6.5; 64 of K 256, N 128 4.5 / 3.7
//
// Past 4608 columns chunks follow each other:
//   K  5120  N 6144   1 12.6 / 14.7    32 15.1 / 18.5   64 22.0 / 29.6      N 1024 16 7.1 / 7.6   N 4096 16 10.4 / 9.9
//   K 12288  N 4096   1 20.8 / 20.0    32 27.9 / 25.3   64 65.2 / 41.4      N 6144 64 66 / 57
//
// Whole chunks for all eight waves have a form of their own (plain_rows_kernel), which keeps more on its way.  linear_kernel, or the form that waits for all loads at every chunk / here:
//   K  6144  N 2048   1  9.9 / 7.8     16 10.9 / 9.5       N 6144  1 18.2 / 16.3    16 22.1 / 20.8      N 8192  1 22.2 / 19.9   8 22.5 / 20.7   16 22.8 / 23.6
//   K  8192  N 2048   1 11.0 / 8.5     16 14.0 / 11.6      N 8192  1 28.2 / 26.1    16 28.1 / 28.4
//   K 10240  N 2048   1 12.5 / 10.3    16 16.1 / 14.5      N 8192  1 32.2 / 30.2     8 32.8 / 31.6
//   K 12288  N 2048   1 14.3 / 11.7    16 18.4 / 16.0      N 6144  1 32.2 / 30.4    16 38.8 / 37.3
//   K 14336  N 2048   1 16.2 / 13.6    16 21.0 / 18.7
//   K 16384  N 4096   1 28.4 / 25.9    16 30.2 / 28.8      N 7168  1 44.5 / 44.0     8 45.3 / 47.0   16 46.1 / 46.0      N 8192  1 50.4 / 49.8   8 51.0 / 51.3
// (Longer ones are not measured.)
static bool whole_chunks(int K) { return K % 2048 == 0 && K >= 6144 && K <= 16384; }

template <class F>
static int with_chunks(int K, F&& launch_with) {   // K: whole_chunks
  switch (K >> 11) {
    case 3: return launch_with(std::integral_constant<int, 3>{});
    case 4: return launch_with(std::integral_constant<int, 4>{});
    case 5: return launch_with(std::integral_constant<int, 5>{});
    case 6: return launch_with(std::integral_constant<int, 6>{});
    case 7: return launch_with(std::integral_constant<int, 7>{});
    default: return launch_with(std::integral_constant<int, 8>{});
  }
}

bool plain_rows_fit(int M, int N, int K, int groups) {
  const int64_t slabs = (int64_t)(N >> 4) * groups;
  if (M > 64) return false;
  if (whole_chunks(K) && M <= 16) return slabs <= (M <= 8 ? 512 : 384);
  if (K > 4608) {
    if (M > 32) return slabs <= (K > 8192 ? 384 : 256);
    return slabs <= 256 && (slabs * ((M + 15) >> 4) >= 192 || (slabs <= 96 && K % 2048 == 0));   // (fewer: linear_kernel's eight waves are level, and ahead where a chunk is not whole)
  }
  if (M <= 16) return K <= 2048 || slabs <= 512;
  if (M <= 32) return K <= 256 || slabs <= (K <= 512 ? 1024 : K <= 1024 ? 512 : 256);
  const int blocks = (N + 63) >> 6, launched = blocks < 8 ? blocks : (blocks + 7) / 8 * 8;
  if (groups > 1 && K <= 128) return slabs <= 1280 || launched * 2 >= blocks * 3;
  return slabs <= (groups > 1 && K <= 256 ? 512 : K <= 512 ? 384 : 256);
}

// Row tiles share a workgroup (and its weights) once there are more workgroups than compute units.  Waves and k-steps a wave by the length of K: four to nine
// k-steps a wave keep all of its part in flight; past 4608 columns chunks follow each other.
template <int EPI>
static int plain_rows_epi(const vmi_hy_linear_args& p, hipStream_t st) {
  const int nks = p.K >> 5, slabs = p.N >> 4;
  auto go = [&](auto* fn, int rw, int j, int mt) {
    return launch(fn, p, dim3(blocks8(slabs), (p.M + 16 * mt - 1) / (16 * mt), p.groups), 64 * rw, (size_t)rw * plain_stride(j, mt), st);
  };
  if ((int64_t)slabs * p.groups * ((p.M + 15) >> 4) <= 256 || p.M <= 16) {
    if (nks <= 4) return go(plain_rows_kernel<4, 1, 1, 1, EPI>, 4, 1, 1);
    if (nks <= 8) return go(plain_rows_kernel<4, 2, 1, 1, EPI>, 4, 2, 1);
    if (nks <= 16) return go(plain_rows_kernel<4, 4, 1, 1, EPI>, 4, 4, 1);
    if (nks <= 32) return go(plain_rows_kernel<8, 4, 1, 1, EPI>, 8, 4, 1);
    if (nks <= 64) return go(plain_rows_kernel<8, 8, 1, 1, EPI>, 8, 8, 1);
    if (nks <= 96) return go(plain_rows_kernel<16, 6, 1, 1, EPI>, 16, 6, 1);
    if (nks <= 128) return go(plain_rows_kernel<16, 8, 1, 1, EPI>, 16, 8, 1);
    if (nks <= 144) return go(plain_rows_kernel<16, 9, 1, 1, EPI>, 16, 9, 1);
    auto whole = [&](auto chunks) {   // (requests for rows: 2, 8 or 16 of them)
      constexpr int NCH = decltype(chunks)::value;
      if (p.M <= 2) return go(plain_rows_kernel<8, 8, 1, 3, EPI, NCH, 1>, 8, 8, 1);
      if (p.M <= 8) return go(plain_rows_kernel<8, 8, 1, 3, EPI, NCH, 4>, 8, 8, 1);
      return go(plain_rows_kernel<8, 8, 1, 3, EPI, NCH, 8>, 8, 8, 1);
    };
    if (whole_chunks(p.K)) return with_chunks(p.K, whole);
    return go(plain_rows_kernel<8, 8, 1, 3, EPI>, 8, 8, 1);
  }
  if (nks <= 4) return go(plain_rows_kernel<4, 1, 2, 1, EPI>, 4, 1, 2);
  if (nks <= 8) return go(plain_rows_kernel<4, 2, 2, 1, EPI>, 4, 2, 2);
  if (nks <= 16) return go(plain_rows_kernel<4, 4, 2, 1, EPI>, 4, 4, 2);
  if (nks <= 32) return go(plain_rows_kernel<8, 4, 2, 1, EPI>, 8, 4, 2);
  if (nks <= 64) return go(plain_rows_kernel<16, 4, 2, 1, EPI>, 16, 4, 2);
  return go(plain_rows_kernel<16, 4, 2, 2, EPI>, 16, 4, 2);
}

// linear_kernel / here, us, weights not in the Infinity Cache: K 512, N 256 1 / 16 rows 3.5 / 4.4 -> 2.1 / 2.4, K 2048, N 1024 4.5 / 5.8 -> 3.3 / 4.1, N 4096 7.5 / 10.3 -> 5.7 / 6.7; K 4096, N 2048 8.3 / 12.0 -> 6.4 / 8.9; K 8192, N
// 4096 1 / 8 19.0 / 25.0 -> 15.2 / 16.7, K 12288, N 6144 34.9 / 46.6 -> 31.5 / 38.3; K 10240, N 5120 26.2 / 36.7 -> 23.5 / 29.4, K 16384, N 8192 53.8 / 65.7 -> 51.0 / 55.0.  (Past 16 rows linear_kernel, as before.)
bool concat_rows_fit(int M, int N, int K) {
  if (M > 16) return false;
  return whole_chunks(K) ? M <= 8 && N <= 16 * 512 : K <= 4608 && plain_rows_fit(M, N, K, 1);   // (registers hold four requests of float32 rows three chunks ahead, not eight)
}

int launch_concat_rows(const vmi_hy_linear_args& p, hipStream_t st) {
  constexpr int EPI = VMI_HY_E_FLOAT, XK = VMI_HY_X_CONCAT;
  const int nks = p.K >> 5;
  auto go = [&](auto* fn, int rw, int j) { return launch(fn, p, dim3(blocks8(p.N >> 4), 1, 1), 64 * rw, (size_t)rw * plain_stride(j, 1), st); };
  if (nks <= 16) return go(plain_rows_kernel<4, 4, 1, 1, EPI, 0, 4, XK>, 4, 4);
  if (nks <= 32) return go(plain_rows_kernel<8, 4, 1, 1, EPI, 0, 4, XK>, 8, 4);
  if (nks <= 64) return go(plain_rows_kernel<8, 8, 1, 1, EPI, 0, 8, XK>, 8, 8);
  if (nks <= 96) return go(plain_rows_kernel<16, 6, 1, 1, EPI, 0, 6, XK>, 16, 6);
  if (nks <= 144) return go(plain_rows_kernel<16, 9, 1, 1, EPI, 0, 9, XK>, 16, 9);
  auto whole = [&](auto chunks) {
    constexpr int NCH = decltype(chunks)::value;
    return p.M <= 2 ? go(plain_rows_kernel<8, 8, 1, 3, EPI, NCH, 1, XK>, 8, 8) : go(plain_rows_kernel<8, 8, 1, 3, EPI, NCH, 4, XK>, 8, 8);
  };
  return with_chunks(p.K, whole);
}

// Whether a product is one of plain_rows_kernel's with four waves: of up to 64 rows, K up to 512, as plain_rows_epi has them
static bool beside_fits(const vmi_hy_linear_args& p, const vmi_hy_step& s) {
  return p.dtype == VMI_HY_BF16 && p.x_kind == VMI_HY_X_ROWS && p.epilogue == VMI_HY_E_STORE && (p.K >> 5) <= 16 && !group_tiles_fit(p) && plain_rows_fit(p.M, p.N, p.K, p.groups) &&
         s.T <= 4096;
}
template <class Prep>
static int launch_beside(const vmi_hy_linear_args& p, const Prep& prep, const vmi_hy_step& s, size_t prep_lds, const char* who, hipStream_t st) {
  const int nks = p.K >> 5, slabs = blocks8(p.N >> 4), mt = (int64_t)(p.N >> 4) * p.groups * ((p.M + 15) >> 4) <= 256 || p.M <= 16 ? 1 : 2, blocks = (p.M + 16 * mt - 1) / (16 * mt);
  auto go = [&](auto* fn, int j) {
    const size_t lds = std::max((size_t)4 * plain_stride(j, mt), prep_lds);
    if (int rc = allow_lds(fn, lds, who)) return rc;
    hipLaunchKernelGGL(fn, dim3(s.T + slabs * blocks * p.groups), dim3(256), lds, st, p, prep, s, slabs, blocks);
    return launched(who);
  };
  if (nks <= 4) return mt == 1 ? go(rows_beside_kernel<1, 1, Prep>, 1) : go(rows_beside_kernel<1, 2, Prep>, 1);
  if (nks <= 8) return mt == 1 ? go(rows_beside_kernel<2, 1, Prep>, 2) : go(rows_beside_kernel<2, 2, Prep>, 2);
  return mt == 1 ? go(rows_beside_kernel<4, 1, Prep>, 4) : go(rows_beside_kernel<4, 2, Prep>, 4);
}

int launch_latent_prompt_in(const vmi_hy_linear_args& l, const vmi_hy_latent_prep_args& a, void* rows, int row0, bool mixed, const vmi_hy_step& s, hipStream_t st, const char* who) {
  if (beside_fits(l, s)) return launch_beside(l, LatentPromptPrep{a, static_cast<b16*>(rows), row0, mixed}, s, latent_prep_lds(a.rot_n), who, st);
  if (int rc = vmi_hy_linear(&l, st)) return rc;
  return launch_latent_prompt_prep(a, rows, row0, mixed, s, st, who);
}

int launch_plain_rows(const vmi_hy_linear_args& p, hipStream_t st) {
  switch (p.epilogue) {
    case VMI_HY_E_STORE: return plain_rows_epi<VMI_HY_E_STORE>(p, st);
    case VMI_HY_E_RESIDUAL: return plain_rows_epi<VMI_HY_E_RESIDUAL>(p, st);
    default: return plain_rows_epi<VMI_HY_E_GATED>(p, st);
  }
}

}  // namespace vmi_hybrid

using namespace vmi_hybrid;

extern "C" {

int vmi_hy_latent_in(const vmi_hy_linear_args* l, const vmi_hy_latent_prep_args* a, const vmi_hy_step* s, void* stream) {
  static const char* who = "vmi_hy_latent_in";
  if (int rc = check_linear(l, who)) return rc;
  if (int rc = check_latent_prep(a, s, who)) return rc;
  if (a->dtype != l->dtype || a->device != l->device || !beside_fits(*l, *s)) {
    if (int rc = vmi_hy_linear(l, stream)) return rc;
    return vmi_hy_latent_prep(a, s, stream);
  }
  DeviceScope dev(l->device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  return launch_beside(*l, LatentPrep{*a}, *s, latent_prep_lds(a->rot_n), who, static_cast<hipStream_t>(stream));
}

int vmi_hy_kv_prep_in(const vmi_hy_linear_args* l, const vmi_hy_kv_prep_args* a, const vmi_hy_step* s, void* stream) {
  static const char* who = "vmi_hy_kv_prep_in";
  if (int rc = check_linear(l, who)) return rc;
  if (int rc = check_kv_prep(a, s, who)) return rc;
  if (a->dtype != l->dtype || a->device != l->device || !beside_fits(*l, *s)) {
    if (int rc = vmi_hy_linear(l, stream)) return rc;
    return vmi_hy_kv_prep(a, s, stream);
  }
  DeviceScope dev(l->device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  return launch_beside(*l, KvPrep{*a}, *s, 0, who, static_cast<hipStream_t>(stream));
}

}  // extern "C"
