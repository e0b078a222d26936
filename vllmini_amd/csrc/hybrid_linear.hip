// The linear layers and the elementwise ends of a step (include/vmi_hybrid.h).
//
// y = epilogue(prologue(x) . W^T), written for steps of few rows, where the weights are what has to be read: every wave owns 16
// output columns and streams its weight tiles (one contiguous KiB per k-step of 32) straight into registers one or two chunks ahead; the
// BM rows of x go through LDS in chunks of K, double-buffered, normalised / concatenated / rounded to the element type on their
// way in, so few rows need no normalised copy of the residual stream (norm_first: when they are better written once).  KS > 1: the k-steps of a chunk are dealt over KS waves
// whose partial tiles meet in LDS in a fixed order.  D[row = column n][col = row m]: a lane ends with 4 consecutive columns of
// one row, so every epilogue works on vectors.
#include <string>

#include "hybrid_common.hpp"
#include "hybrid_linear.hpp"
#include "step_inputs.hpp"

namespace vmi_hybrid {

static thread_local std::string g_err;
int fail(int code, const char* who, const char* what) {
  g_err.assign(who);
  g_err.append(": ");
  g_err.append(what);
  return code;
}
int launched(const char* who) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? VMI_HY_OK : fail(VMI_HY_E_HIP, who, hipGetErrorString(e));
}

template <typename T, int BM, int KS>
struct Chunk {
  static constexpr bool DEEP = BM == 16 && sizeof(T) == 2;   // few rows: bytes in flight are what counts
  static constexpr int CS = DEEP && KS < 8 ? 8 : 4;                    // k-steps a wave takes from a chunk
  static constexpr int NB = DEEP ? 3 : 2;                     // chunks of weights in registers, NB - 1 of them ahead
  static constexpr int KC = 32 * CS * KS;                     // columns of x in a chunk
};

// 8 consecutive elements of row m at column k, as they go into LDS
template <typename T, int XK>
struct XUnit;
template <typename T>
struct XUnit<T, VMI_HY_X_ROWS> {
  V8<T> v = zero8<T>();
  __device__ __forceinline__ void load(const vmi_hy_linear_args& p, int64_t row, int64_t goff, int k) {
    v = load8(static_cast<const T*>(p.x) + goff + row * p.ldx + k);
  }
  __device__ __forceinline__ V8<T> finish(const float*, int, float, float) const { return v; }
};
template <typename T>
struct XUnit<T, VMI_HY_X_NORM> {
  f32x8 v = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  __device__ __forceinline__ void load(const vmi_hy_linear_args& p, int64_t row, int64_t, int k) {
    v = load8(static_cast<const float*>(p.x) + row * p.ldx + k);
  }
  __device__ __forceinline__ V8<T> finish(const float* nw, int k, float mean, float rstd) const {
    const f32x8 w = load8(nw + k);   // (zero past norm_n: padding columns come out as zeros)
    f32x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (v[e] - mean) * rstd * w[e];
    return from_f32<T>(r);
  }
};
template <typename T>
struct XUnit<T, VMI_HY_X_CONCAT> {
  f32x8 v = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  __device__ __forceinline__ void load(const vmi_hy_linear_args& p, int64_t row, int64_t, int k) {
    const int half = p.K >> 1;
    const float* src = static_cast<const float*>(k < half ? p.x : p.x2);
    v = load8(src + row * p.ldx + (k < half ? k : k - half));
  }
  __device__ __forceinline__ V8<T> finish(const float*, int, float, float) const { return from_f32<T>(v); }
};

template <typename T, int BM, int NW, int KS, int XK, int EPI>
__global__ __launch_bounds__(NW* KS * 64) void linear_kernel(const vmi_hy_linear_args p) {
  using CK = Chunk<T, BM, KS>;
  constexpr int TH = NW * KS * 64, MT = BM / 16, CS = CK::CS, KC = CK::KC, NB_W = CK::NB;
  constexpr int LD = KC + 16 / (int)sizeof(T), UPR = KC / 8, UPT = BM * UPR / TH;
  static_assert(BM * UPR % TH == 0, "a chunk's units divide over the threads");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T* xs = reinterpret_cast<T*>(smem);                                   // [2][BM][LD]
  float* stats = reinterpret_cast<float*>(xs + (size_t)2 * BM * LD);    // [BM][2]
  float* red = stats + 2 * BM;                                          // [KS - 1][NW][MT][64][4]
  // the norm's weight, in LDS: read from memory between the weight tiles it would wait for all of them
  float* nwl = red + (KS - 1) * NW * MT * 256;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = wave % NW, ks = wave / NW;
  const int kc = lane >> 4, r16 = lane & 15;
  // column blocks are dealt so that all row blocks of one stay on one XCD (workgroups go round-robin over the 8 of them): its
  // weights are read from HBM once
  const int MB = (p.M + BM - 1) / BM, NB = (p.N + 16 * NW - 1) / (16 * NW);
  // (fewer than 8 of them: a plain order, or most XCDs would stay idle)
  const int grp = blockIdx.y;
  const int nb = NB < 8 ? (int)blockIdx.x % NB : (int)(blockIdx.x / (8 * MB)) * 8 + (int)(blockIdx.x & 7);
  const int mb = NB < 8 ? (int)blockIdx.x / NB : (int)(blockIdx.x >> 3) % MB;
  if (nb >= NB) return;
  const int m0 = mb * BM, n0 = (nb * NW + nw) * 16, nks = p.K >> 5;
  const bool nvalid = n0 < p.N;
  const int64_t goff = (int64_t)grp * p.x_gstride;

  const T* wp = static_cast<const T*>(p.w) + (((int64_t)grp * (p.N >> 4) + (nvalid ? n0 >> 4 : 0)) * nks * 64 + lane) * 8;
  const int nchunk = (p.K + KC - 1) / KC;
  V8<T> wb[NB_W][CS];
  auto load_w = [&](V8<T>(&dst)[CS], int c) {
#pragma unroll
    for (int j = 0; j < CS; ++j) {
      // (no lane-wise condition around a load, here or for x: all of a chunk's are in flight together.  A k-step past the last
      //  one reads that one again and meets zeros of x)
      const int k = min(c * (CS * KS) + ks * CS + j, nks - 1);
      dst[j] = load8(wp + (int64_t)k * 512);
    }
  };
#pragma unroll
  for (int b = 0; b < NB_W - 1; ++b) load_w(wb[b], b);

  auto source_row = [&](int m) -> int64_t {
    const int mm = m0 + m < p.M ? m0 + m : p.M - 1;
    if constexpr (XK == VMI_HY_X_NORM) return p.rows ? p.rows[mm] : mm;
    return mm;
  };

  if constexpr (XK == VMI_HY_X_NORM) {   // row statistics, one pass around the row's first element: no cancellation to speak of
    constexpr int NWV = TH / 64;
    const int mrows = min(BM, p.M - m0);
    for (int k = tid * 4; k < p.K; k += TH * 4) *reinterpret_cast<f32x4*>(nwl + k) = *reinterpret_cast<const f32x4*>(p.norm_w + k);
    for (int mbase = wave; mbase < mrows; mbase += 4 * NWV) {
      const float* row[4];
      float sh[4], s[4], q[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = mbase + i * NWV < mrows ? mbase + i * NWV : mbase;
        row[i] = static_cast<const float*>(p.x) + source_row(m) * p.ldx;
        sh[i] = p.rms ? 0.f : row[i][0];
        s[i] = q[i] = 0.f;
      }
      for (int k = lane * 4; k < p.K; k += 256) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(row[i] + k);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float d = k + e < p.norm_n ? v[e] - sh[i] : 0.f;
            s[i] += d;
            q[i] = fmaf(d, d, q[i]);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float ms = p.rms ? 0.f : wave_sum(s[i]) / (float)p.norm_n, mq = wave_sum(q[i]) / (float)p.norm_n;
        const int m = mbase + i * NWV;
        if (lane == 0 && m < mrows) {
          stats[2 * m] = sh[i] + ms;
          stats[2 * m + 1] = 1.f / sqrtf(fmaxf(mq - ms * ms, 0.f) + p.eps);
        }
      }
    }
    __syncthreads();
  }

  int64_t srow[UPT];
  int xm[UPT], xk[UPT];
  bool xin[UPT];
  float mean[UPT], rstd[UPT];
#pragma unroll
  for (int i = 0; i < UPT; ++i) {
    const int u = tid + i * TH;
    xm[i] = u / UPR;
    xk[i] = (u % UPR) * 8;
    srow[i] = source_row(xm[i]);
    xin[i] = m0 + xm[i] < p.M;
    mean[i] = rstd[i] = 0.f;
    if (XK == VMI_HY_X_NORM && xin[i]) {
      mean[i] = stats[2 * xm[i]];
      rstd[i] = stats[2 * xm[i] + 1];
    }
  }
  XUnit<T, XK> xu[UPT];
  auto load_x = [&](int c) {
#pragma unroll
    for (int i = 0; i < UPT; ++i)   // (a wave whose rows all lie past M reads none: a scalar condition)
      if ((wave * 64 + i * TH) / UPR < p.M - m0) xu[i].load(p, srow[i], goff, min(c * KC + xk[i], p.K - 8));
  };
  load_x(0);

  f32x4 acc[MT];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) acc[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int c, V8<T>(&cur)[CS], V8<T>(&nxt)[CS]) {
    T* dst = xs + (size_t)(c & 1) * BM * LD;
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const int k = c * KC + xk[u];
      const V8<T> v = xu[u].finish(nwl, min(k, p.K - 8), mean[u], rstd[u]);
      *reinterpret_cast<V8<T>*>(dst + xm[u] * LD + xk[u]) = xin[u] && k < p.K ? v : zero8<T>();
    }
    // x first, and the weights whatever is left (past the end: one tile again, a cache hit): a wait for x then always knows how
    // many younger loads it may leave in flight
    if (c + 1 < nchunk) load_x(c + 1);
    load_w(nxt, c + NB_W - 1);
    __syncthreads();   // (two buffers: the writes of chunk c + 1 go where chunk c - 1 was read, which every wave has left behind)
#pragma unroll
    for (int j = 0; j < CS; ++j)
#pragma unroll
      for (int mi = 0; mi < MT; ++mi) mma(acc[mi], cur[j], load8(dst + (mi * 16 + r16) * LD + (ks * CS + j) * 32 + 8 * kc));
  };
  for (int c = 0; c < nchunk; c += NB_W) {   // chunk c sits in wb[c % NB_W]; the one behind it has been used up
#pragma unroll
    for (int b = 0; b < NB_W; ++b)
      if (c + b < nchunk) step(c + b, wb[b], wb[(b + NB_W - 1) % NB_W]);
  }

  if constexpr (KS > 1) {
    if (ks > 0) {
#pragma unroll
      for (int mi = 0; mi < MT; ++mi)
        *reinterpret_cast<f32x4*>(red + ((((ks - 1) * NW + nw) * MT + mi) * 64 + lane) * 4) = acc[mi];
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int s = 1; s < KS; ++s)
#pragma unroll
      for (int mi = 0; mi < MT; ++mi)
        acc[mi] += *reinterpret_cast<const f32x4*>(red + ((((s - 1) * NW + nw) * MT + mi) * 64 + lane) * 4);
  }
  if (!nvalid) return;

#pragma unroll
  for (int mi = 0; mi < MT; ++mi) {
    const int m = m0 + mi * 16 + r16;
    if (m < p.M) epilogue<T, EPI>(p, acc[mi], m, n0 + 4 * kc, n0, grp);
  }
}

// Steps of few rows behind a norm whose x fits a compute unit's LDS (bfloat16, one group).  Such a product is the reading of its weights, so nothing but
// that reading may take time:
//   * a workgroup puts all rows of x into LDS once, normed and rounded on the way: every wave has a share of a row and all of
//     its loads in flight; after that the walk over K has no barrier and no load but the weights';
//   * then it walks over slabs of 16 columns, blockIdx, blockIdx + grid, ..: its W waves take a W-th of K each and the ring of weight
//     tiles runs on across slabs; a slab's partial tiles meet in LDS (two places, one barrier a slab) and one wave, another each time,
//     adds them in a fixed order and stores;
//   * rows past M repeat the last one: their results go nowhere.
// In linear_kernel x comes in chunks of K behind a barrier each, and ONE wave makes a row's statistics in front of everything, behind the first
// weights.  One row, K 4096: N 24576 57.4 -> 37.1 us (5.4 TB/s), N 8192 25.6 -> 17.1; K 1024: N 6144 10.1 -> 7.7, N 50272 30.6 -> 22.0; 16 rows, K 4096,
// N 24576 67.6 -> 46.6; 32 rows, K 2048: N 22528 40.4 -> 29.9, N 50272 85.8 -> 51.9.  (Non-temporal loads of the weights: 36.5, but 77 against 74 us
// for 412 MB and slower wherever they stay in the Infinity Cache.  16 waves a workgroup where there is one slab a compute unit: 9.9 -> 11.3.)
// NCH > 0: rows of 1024 NCH columns, NCH whole chunks a wave.  Then nothing in the walk depends on a condition but its end and the stores: the compiler counts loads in
// flight, and where paths meet that differ in them it waits for all of them, every NB chunks.  General form -> this one, weights not in the Infinity Cache, us: K 4096, N 4096 1 / 4 / 8
// rows 11.1 / 12.5 / 14.8 -> 8.8 / 11.0 / 13.1, N 8192 16.7 / 17.8 / 21.2 -> 14.5 / 16.8 / 20.1, N 24576 38.5 / 39.0 / 43.1 -> 37.1 / 38.4 / 41.9, N 50272 72.9 -> 71.8; K 2048, N 12288 1 / 16 rows 13.8 / 15.4 -> 11.8 /
// 14.4, N 50272 40.3 / 44.8 -> 37.8 / 43.3; K 1024, N 50272 22.3 / 23.1 -> 20.6 / 22.0.  (201 and 412 MB alone, nothing computed: 34.5 and 70.)
template <int MT, int W, int PL, int CU, int EPI, int NCH = 0>
__global__ __launch_bounds__(64 * W, 2 * CU) void resident_kernel(const vmi_hy_linear_args p, const int slabs) {
  constexpr int CS = 4, NB = CU > 1 ? 4 : 6;   // k-steps of a chunk, chunks of weights in registers (NB - 1 of them ahead)
  constexpr int KS = NCH * CS;                 // k-steps of a wave
  if constexpr (NCH > 0) need(p.x), need(p.ldx), need(p.rows), need(p.norm_w), need(p.norm_n), need(p.rms), need(p.eps), need(p.w), need(p.y), need(p.ldy), need(p.M), need(p.N), need(p.K);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int LD = p.K + 8, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kc = lane >> 4, r16 = lane & 15;
  f32x4* red = reinterpret_cast<f32x4*>(smem);                         // [PL][W - 1][MT][64]
  float* part = reinterpret_cast<float*>(red + PL * (W - 1) * MT * 64);       // [W][2] parts of a row's sums
  b16* xs = reinterpret_cast<b16*>(part + 2 * W);                      // [M][LD]
  const int nks = p.K >> 5, kpw = (nks + W - 1) / W, nch = (kpw + CS - 1) / CS;
  const int mine = (slabs - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x, total = mine * nch;   // slabs, chunks of this workgroup

  b16x8 wb[NB][CS];
  const b16* wp = static_cast<const b16*>(p.w) + lane * 8;
  int ls = blockIdx.x, lc = 0;   // the chunk to load next: slab and chunk of it
  // whole chunks: chunk c of slab ls.  Past the last slab 16 bytes of one for all lanes, which meet nothing; requests stay in the order of their use
  [[maybe_unused]] auto load_whole = [&](b16x8(&dst)[CS], int c) {
    const bool past = ls >= slabs;
    const b16* at = static_cast<const b16*>(p.w) + ((int64_t)(past ? (int)blockIdx.x : ls) * (W * KS) + wave * KS + c * CS) * 512 + (past ? 0 : lane * 8);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < CS; ++j) dst[j] = load8(at + j * 512);
    __builtin_amdgcn_sched_barrier(0);
    if (c == NCH - 1) ls += gridDim.x;
  };
  auto load_w = [&](b16x8(&dst)[CS]) {
    const b16* at = wp + (int64_t)ls * nks * 512;
#pragma unroll
    for (int j = 0; j < CS; ++j) dst[j] = load8(at + (int64_t)min(wave * kpw + min(lc * CS + j, kpw - 1), nks - 1) * 512);
    if (lc + 1 < nch) {
      ++lc;
    } else if (ls + (int)gridDim.x < slabs) {   // (past the last chunk: that one again, a cache hit)
      lc = 0;
      ls += gridDim.x;
    }
  };

  // x into LDS: wpr waves a row, rpp rows at a time
  const int M = p.M, upr = p.K >> 3;
  const int wpr = M == 1 ? W : M == 2 ? W / 2 : M <= 4 ? W / 4 : M <= 8 ? W / 8 : 1, rpp = W / wpr, sub = wave % wpr, step8 = 64 * wpr;
  const int u0 = sub * 64 + lane;   // this lane's units of a row of its wave: u0, u0 + step8, ..
  auto row_at = [&](int round) { return min(round * rpp + wave / wpr, M - 1); };
  const int rounds = (M + rpp - 1) / rpp;
  auto open_ring = [&]() {
#pragma unroll
    for (int b = 0; b < NB - 1; ++b) {
      if constexpr (NCH > 0) load_whole(wb[b], b % NCH);
      else load_w(wb[b]);
    }
  };
  {
    constexpr int HOLD = CU > 1 ? 2 : 4;   // units of 8 columns a lane keeps; longer shares are read again
    f32x8 w[HOLD];
    f32x8 v[HOLD];
    float sh;
    const float* row;
    auto fetch = [&](int round) {
      const int m = row_at(round);
      row = static_cast<const float*>(p.x) + (p.rows ? p.rows[m] : m) * p.ldx;
      sh = p.rms ? 0.f : row[0];
#pragma unroll
      for (int i = 0; i < HOLD; ++i) v[i] = load8(row + min(u0 + i * step8, upr - 1) * 8);
    };
    fetch(0);
#pragma unroll
    for (int i = 0; i < HOLD; ++i) w[i] = load8(p.norm_w + min(u0 + i * step8, upr - 1) * 8);
    open_ring();   // (behind the first loads of x, so that waiting for those leaves the weights in flight)
    auto one_round = [&](int round) {
      float s = 0.f, q = 0.f;
      auto sums = [&](const f32x8& x, int u) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = u * 8 + e < p.norm_n ? x[e] - sh : 0.f;
          s += d;
          q = fmaf(d, d, q);
        }
      };
#pragma unroll
      for (int i = 0; i < HOLD; ++i)
        if (u0 + i * step8 < upr) sums(v[i], u0 + i * step8);
      for (int u = u0 + HOLD * step8; u < upr; u += step8) sums(load8(row + u * 8), u);
      s = wave_sum(s);
      q = wave_sum(q);
      if (wpr > 1) {
        if (lane == 0) part[2 * wave] = s, part[2 * wave + 1] = q;
        __syncthreads();
        s = q = 0.f;
        for (int i = 0; i < wpr; ++i) s += part[2 * (wave - sub + i)], q += part[2 * (wave - sub + i) + 1];
        if (round + 1 < rounds) __syncthreads();
      }
      const float ms = p.rms ? 0.f : s / (float)p.norm_n, mean = sh + ms;
      const float rstd = 1.f / sqrtf(fmaxf(q / (float)p.norm_n - ms * ms, 0.f) + p.eps);
      b16* to = xs + row_at(round) * LD;
      auto put = [&](const f32x8& x, const f32x8& g, int u) {
        f32x8 r;
#pragma unroll
        for (int e = 0; e < 8; ++e) r[e] = (x[e] - mean) * rstd * g[e];   // (the weight is zero past norm_n)
        *reinterpret_cast<b16x8*>(to + u * 8) = from_f32<b16>(r);
      };
#pragma unroll
      for (int i = 0; i < HOLD; ++i)
        if (u0 + i * step8 < upr) put(v[i], w[i], u0 + i * step8);
      for (int u = u0 + HOLD * step8; u < upr; u += step8) put(load8(row + u * 8), load8(p.norm_w + u * 8), u);
    };
    // (by itself: with the following ones, whose rows come behind the weights, it would wait for those; and what came in front of the weights is there, whichever lanes use it)
    constexpr int RING = (NB - 1) * CS;
    __builtin_amdgcn_s_waitcnt(0x0f70 | (RING & 15) | (RING >> 4 << 14));   // vmcnt(RING)
    one_round(0);
    for (int round = 1; round < rounds; ++round) {
      fetch(round);
      one_round(round);
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    }
  }
  __syncthreads();

  const b16* xa[MT];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) xa[mi] = xs + min(mi * 16 + r16, M - 1) * LD + 8 * kc;
  f32x4 acc[MT];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) acc[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
  int slab = blockIdx.x, c = 0, i = 0;   // of the chunk to multiply next; slabs done
  auto meet = [&]() {   // a slab's partial tiles
    f32x4* to = red + (PL > 1 ? (i & 1) * (W - 1) * MT * 64 : 0);
    const int behind = (wave - i) & (W - 1);   // 0: the wave that adds up; the others' places in their order behind it
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
      if (behind) to[((behind - 1) * MT + mi) * 64 + lane] = acc[mi];
    __syncthreads();   // (two places: who still adds up slab i has not passed the barrier of slab i + 1; one: a second barrier)
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
      if (behind == 0) {
#pragma unroll
        for (int w = 0; w < W - 1; ++w) acc[mi] += to[(w * MT + mi) * 64 + lane];
        if (mi * 16 + r16 < M) epilogue<b16, EPI>(p, acc[mi], mi * 16 + r16, slab * 16 + 4 * kc, slab * 16, 0);
      }
      acc[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (PL == 1) __syncthreads();
    ++i;
    slab += gridDim.x;
  };
  [[maybe_unused]] auto step = [&](b16x8(&cur)[CS], b16x8(&nxt)[CS]) {
    load_w(nxt);
#pragma unroll
    for (int j = 0; j < CS; ++j) {
      const int kk = c * CS + j, k = wave * kpw + kk;
      if (kk < kpw && k < nks) {   // (scalar)
#pragma unroll
        for (int mi = 0; mi < MT; ++mi) mma(acc[mi], cur[j], load8(xa[mi] + k * 32));
      }
    }
    if (++c < nch) return;
    meet();
    c = 0;
  };
  if constexpr (NCH == 0) {
    for (int t = 0; t < total; t += NB) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (t + b < total) step(wb[b], wb[(b + NB - 1) % NB]);
    }
  } else {
    // a slab whose first chunk is in place B0 of the ring; more: its chunks' successors are asked for
    auto walk = [&](auto b0, bool more) {
      constexpr int B0 = decltype(b0)::value;
#pragma unroll
      for (int n = 0; n < NCH; ++n) {
        if (more) load_whole(wb[(B0 + n + NB - 1) % NB], (n + NB - 1) % NCH);
#pragma unroll
        for (int j = 0; j < CS; ++j)
#pragma unroll
          for (int mi = 0; mi < MT; ++mi) mma(acc[mi], wb[B0 + n][j], load8(xa[mi] + (wave * KS + n * CS + j) * 32));
      }
      meet();
    };
    constexpr int ROUND = NB / NCH;   // slabs the ring goes round in
    static_assert(NB % NCH == 0 && ROUND <= 4, "a chunk's place in its slab follows from its place in the ring");
    // whole rounds, then what is left, which the ring holds; one way out of the loop, since any other joins the way back in the compiler's eyes
    for (; slab + (ROUND - 1) * (int)gridDim.x < slabs;) {
      walk(std::integral_constant<int, 0>{}, true);
      if constexpr (ROUND > 1) walk(std::integral_constant<int, NCH % NB>{}, true);
      if constexpr (ROUND > 2) walk(std::integral_constant<int, 2 * NCH % NB>{}, true);
      if constexpr (ROUND > 3) walk(std::integral_constant<int, 3 * NCH % NB>{}, true);
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
    }
  }
}

inline size_t resident_lds(int M, int K, int W, int PL) { return (size_t)PL * (W - 1) * ((M + 15) / 16) * 1024 + 8 * W + (size_t)M * (K + 8) * 2; }

// Whether, and how, a product behind a norm runs in resident_kernel.  2: two places for partial tiles and two workgroups a compute unit; 3: one place,
// so that two workgroups still fit; 1: one workgroup, with a longer ring of weights; 0: not at all.  From 17 rows on a workgroup's reading of
// x (32 rows of 1024: 128 KiB) needs enough slabs behind it: 32 rows, N 6144, K 1024 take 13.2 us here and 11.6 in linear_kernel, N 50272 28.4 and
// 43.8.  Rows that need no norm (K 1024 .. 12288, N 1024 .. 4096) stay in linear_kernel, whose waves see x as early: 3.5 us there, 4.5 here
// for one row of 1024, 22.0 and 21.5 for one of 12288.
static int resident_kind(int M, int N, int K) {
  if (M > 32 || K < 256 || (M > 16 && N < 16 * 512)) return 0;
  if (resident_lds(M, K, 8, 2) <= LDS_PER_CU / 2) return 2;
  if (M > 16 && resident_lds(M, K, 8, 1) <= LDS_PER_CU / 2) return 3;
  return resident_lds(M, K, 8, 1) <= LDS_PER_CU ? 1 : 0;
}

// ... and where it does not pay: linear_kernel is as fast or faster on short rows while all of its workgroups are on the chip at once (up to
// 1024 of 32 columns, 2048 to 3072 of 64; in between and beyond it takes another round).  linear_kernel / resident_kernel in us: 8 rows, K 256, N 12288 7.4 / 6.6, N 32768
// 7.1 / 8.4; 16 rows, K 256, N 16384 7.9 / 8.4, N 32768 7.5 / 9.8, K 512, N 32768 10.5 / 10.4; 17 rows, K 512, N 8192 8.0 / 9.3, N 12288 13.6 / 9.6, N 24576 11.2 / 11.6; 32 rows, K 256, N 24576 8.2 / 12.8, K 768, N 16384
// 10.8 / 12.9, K 1024 14.9 / 14.3, K 1280 17.1 / 18.8, K 1536 19.2 / 20.0, K 2048 27.6 / 22.8; N 8192, 17 and 32 rows, K 1024 10.8 / 10.4 and 11.0 / 11.7, K 1536 11.8 / 13.0 and
// 12.1 / 14.0, K 2048 15.4 / 13.8 and 16.0 / 16.4 (a wave takes its share of K four k-steps at a time: multiples of 1024 leave none unused)
static bool resident_pays(int M, int N, int K) {
  const int wgs = (N >> 4) * ((M + 15) >> 4);
  if ((wgs > 1024 && wgs < 2048) || wgs > 3072) return true;
  if (M <= 16) return K > 512 || (M <= 8 && wgs <= 1024);
  return wgs <= 1024 ? K % 1024 == 0 && K <= 2048 && M <= 24 : K == 1024 || K >= 1536;
}

template <int MT, int W, int PL, int CU, int EPI>   // CU workgroups a compute unit
static int launch_resident(const vmi_hy_linear_args& p, hipStream_t st) {
  auto* fn = resident_kernel<MT, W, PL, CU, EPI>;
  if constexpr (CU == 2) {   // (longer rows of 17 and more do not leave room for two workgroups)
    if (p.K == 1024) fn = resident_kernel<MT, W, PL, CU, EPI, 1>;
    if constexpr (MT == 1) {
      if (p.K == 2048) fn = resident_kernel<MT, W, PL, CU, EPI, 2>;
      if (p.K == 4096) fn = resident_kernel<MT, W, PL, CU, EPI, 4>;
    }
  }
  const size_t lds = resident_lds(p.M, p.K, W, PL);
  if (int rc = allow_lds(fn, lds, "vmi_hy_linear")) return rc;
  const int slabs = p.N / 16;
  hipLaunchKernelGGL(fn, dim3(slabs < 256 * CU ? slabs : 256 * CU), dim3(64 * W), lds, st, p, slabs);
  return launched("vmi_hy_linear");
}

// Whether the rows behind a norm are better normed once, by a kernel of their own (2.8 us between two others), than in every workgroup of the product:
// long rows, from 17 of them on, where the workgroups' share of that is 32 rows a column of tiles (except of a vocabulary's columns behind rows that stay
// in LDS), from 9 on where the columns are few.  K 4096, in every workgroup -> once: 32 rows, N 4096 25.0 -> 18.3 us, N 12288 56.3 -> 35.5; 40, N 24576 84.4 ->
// 54.4; 16, N 4096 19.3 -> 16.4, N 24576 50.7 -> 46.8; 8, N 8192 21.8 -> 21.4.  Shorter rows gain less than a launch costs a caller who records no graph
// and waits for his own calls (6 us): 32 rows, K 2048, N 12288 22.4 -> 20.7, K 1024, N 8192 15.0 -> 11.6; a prompt of 35 tokens, width 1024, 1.00 -> 1.06 ms.
static bool norm_first(int M, int N, int K) {
  if (K < 4096) return false;
  if (M > 16) return M > 32 || N < 24576 || resident_kind(M, N, K) == 0;
  return M > 8 && N <= 4 * K;
}

template <typename T, int BM, int NW, int KS, int XK, int EPI>
static int launch_linear(const vmi_hy_linear_args& p, hipStream_t st) {
  constexpr int KC = Chunk<T, BM, KS>::KC, LD = KC + 16 / (int)sizeof(T);
  const size_t lds = (size_t)2 * BM * LD * sizeof(T) + 2 * BM * 4 + (size_t)(KS - 1) * NW * (BM / 16) * 64 * 16 +
                     (XK == VMI_HY_X_NORM ? (size_t)p.K * 4 : 0);
  auto* fn = linear_kernel<T, BM, NW, KS, XK, EPI>;
  if (int rc = allow_lds(fn, lds, "vmi_hy_linear")) return rc;
  const int MB = (p.M + BM - 1) / BM, NB = (p.N + 16 * NW - 1) / (16 * NW);
  hipLaunchKernelGGL(fn, dim3((NB < 8 ? NB : (NB + 7) / 8 * 8) * MB, p.groups), dim3(NW * KS * 64), lds, st, p);
  return launched("vmi_hy_linear");
}

template <typename T, int XK, int EPI>
static int linear_shape(const vmi_hy_linear_args& p, hipStream_t st) {
  // few rows: 16-row tiles; a layer with few columns splits K over the waves of a workgroup so that all compute units read
  const int64_t slabs = (int64_t)(p.N / 16) * p.groups;
  constexpr bool PLAIN = sizeof(T) == 2 && XK == VMI_HY_X_ROWS && (EPI == VMI_HY_E_STORE || EPI == VMI_HY_E_RESIDUAL || EPI == VMI_HY_E_GATED);
  if constexpr (sizeof(T) == 2 && XK == VMI_HY_X_CONCAT && EPI == VMI_HY_E_FLOAT)
    if (p.groups == 1 && concat_rows_fit(p.M, p.N, p.K)) return launch_concat_rows(p, st);
  if constexpr (PLAIN && EPI != VMI_HY_E_RESIDUAL)
    if (group_tiles_fit(p)) return launch_group_tiles(p, st);
  if constexpr (PLAIN)
    if (plain_rows_fit(p.M, p.N, p.K, p.groups)) return launch_plain_rows(p, st);
  if constexpr (sizeof(T) == 2 && XK == VMI_HY_X_NORM) {
    if (p.groups == 1 && norm_slabs(p.M, p.N, p.K)) return launch_norm_rows(p, st);
    switch (p.groups == 1 && resident_pays(p.M, p.N, p.K) ? resident_kind(p.M, p.N, p.K) : 0) {
      case 2: return p.M <= 16 ? launch_resident<1, 8, 2, 2, EPI>(p, st) : launch_resident<2, 8, 2, 2, EPI>(p, st);
      case 3: return launch_resident<2, 8, 1, 2, EPI>(p, st);
      case 1: return p.M <= 16 ? launch_resident<1, 8, 1, 1, EPI>(p, st) : launch_resident<2, 8, 1, 1, EPI>(p, st);
      default: break;
    }
  }
  if (p.M <= 32) {
    const int64_t wgs = slabs * ((p.M + 15) / 16);
    if (wgs >= 2048) return launch_linear<T, 16, 4, 1, XK, EPI>(p, st);
    if (wgs >= 400 || p.K < 256) return launch_linear<T, 16, 2, 2, XK, EPI>(p, st);
    if constexpr (sizeof(T) == 2)
      if (wgs < 192 && p.K >= 1024) return launch_linear<T, 16, 1, 8, XK, EPI>(p, st);
    return launch_linear<T, 16, 1, 4, XK, EPI>(p, st);
  }
  if (p.M <= 96 || slabs / 4 * ((p.M + 63) / 64) < 256) return launch_linear<T, 32, 4, 1, XK, EPI>(p, st);
  return launch_linear<T, 64, 4, 1, XK, EPI>(p, st);
}

// rows that stand in p.x normed: what follows a norm
static int linear_normed(const vmi_hy_linear_args& p, hipStream_t st) {
  if (p.groups == 1 && held_rows_pay(p.M, p.N, p.K, p.epilogue == VMI_HY_E_STORE)) return launch_held_rows(p, st);
  switch (p.epilogue) {
    case VMI_HY_E_STORE: return linear_shape<b16, VMI_HY_X_ROWS, VMI_HY_E_STORE>(p, st);
    case VMI_HY_E_FLOAT: return linear_shape<b16, VMI_HY_X_ROWS, VMI_HY_E_FLOAT>(p, st);
    case VMI_HY_E_GLU: return linear_shape<b16, VMI_HY_X_ROWS, VMI_HY_E_GLU>(p, st);
    case VMI_HY_E_STORE_GLU: return linear_shape<b16, VMI_HY_X_ROWS, VMI_HY_E_STORE_GLU>(p, st);
    default: return fail(VMI_HY_E_ARG, "vmi_hy_linear", "this combination of input and epilogue is not built");
  }
}

template <typename T>
static int linear_kind(const vmi_hy_linear_args& p, hipStream_t st) {
  switch (p.x_kind * 8 + p.epilogue) {
    case VMI_HY_X_ROWS * 8 + VMI_HY_E_STORE: return linear_shape<T, VMI_HY_X_ROWS, VMI_HY_E_STORE>(p, st);
    case VMI_HY_X_ROWS * 8 + VMI_HY_E_RESIDUAL: return linear_shape<T, VMI_HY_X_ROWS, VMI_HY_E_RESIDUAL>(p, st);
    case VMI_HY_X_ROWS * 8 + VMI_HY_E_GATED: return linear_shape<T, VMI_HY_X_ROWS, VMI_HY_E_GATED>(p, st);
    case VMI_HY_X_NORM * 8 + VMI_HY_E_STORE: return linear_shape<T, VMI_HY_X_NORM, VMI_HY_E_STORE>(p, st);
    case VMI_HY_X_NORM * 8 + VMI_HY_E_FLOAT: return linear_shape<T, VMI_HY_X_NORM, VMI_HY_E_FLOAT>(p, st);
    case VMI_HY_X_NORM * 8 + VMI_HY_E_GLU: return linear_shape<T, VMI_HY_X_NORM, VMI_HY_E_GLU>(p, st);
    case VMI_HY_X_NORM * 8 + VMI_HY_E_STORE_GLU: return linear_shape<T, VMI_HY_X_NORM, VMI_HY_E_STORE_GLU>(p, st);
    case VMI_HY_X_CONCAT * 8 + VMI_HY_E_FLOAT: return linear_shape<T, VMI_HY_X_CONCAT, VMI_HY_E_FLOAT>(p, st);
    default: return fail(VMI_HY_E_ARG, "vmi_hy_linear", "this combination of input and epilogue is not built");
  }
}

// ---- elementwise ends ---------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void embed_kernel(const int64_t* __restrict__ ids, const b16* __restrict__ table,
                                                    float* __restrict__ x, int width, int ld, int vocab, float scale) {
  const int t = blockIdx.x;
  int64_t id = ids[t];
  if (id < 0 || id >= vocab) id = 0;   // (ids are checked on the host; sampled ones are in range by construction)
  for (int k = threadIdx.x * 4; k < ld; k += 1024) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = k + e < width ? (float)table[id * (int64_t)ld + k + e] * scale : 0.f;
    *reinterpret_cast<f32x4*>(x + (int64_t)t * ld + k) = o;
  }
}

// One workgroup per row of x, or of its rows[t]; NV times 1024 columns of it stay in registers between the three passes (what a row has beyond them, with NV = 8, is read again).
// All of that, the addend and the norm's weight are asked for at once: with a load, an add and a store to the row a step, each step waited for the one before, and the weight came a
// trip to memory behind the statistics.  us, with an addend, so / here: 60 rows of 1024 / 2048 / 4096 3.9 / 4.0 / 4.7 -> 3.4 / 3.4 / 3.9, 2773 9.8 / 14.0 / 23.6 -> 7.0 / 11.8 / 21.7 (4.4 TB/s).
template <typename T, int NV>
__global__ __launch_bounds__(256) void add_norm_kernel(float* x, int64_t ldx, const int* rows, const T* add, int64_t ld_add,
                                                       const float* norm_w, T* out, int n, int ld, float eps, int rms) {
  __shared__ float part[2][4];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float* row = x + (rows ? rows[t] : t) * ldx;
  f32x4 v[NV], w[NV];
  V4<T> d[NV];
  float s = 0.f;
  auto sum = [&](const f32x4& a, int k) {   // (of the n columns that are normed: what lies behind them may be anything)
    s += (k < n ? a[0] : 0.f) + (k + 1 < n ? a[1] : 0.f) + (k + 2 < n ? a[2] : 0.f) + (k + 3 < n ? a[3] : 0.f);
  };
#pragma unroll
  for (int i = 0; i < NV; ++i) {   // (past the row: its last columns again)
    const int k = min((tid + i * 256) * 4, ld - 4);
    v[i] = *reinterpret_cast<const f32x4*>(row + k);
    if (add) d[i] = *reinterpret_cast<const V4<T>*>(add + (int64_t)t * ld_add + k);
    if (out) w[i] = *reinterpret_cast<const f32x4*>(norm_w + k);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = (tid + i * 256) * 4;
    if (add) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] += (float)d[i][e];
      if (k < ld) *reinterpret_cast<f32x4*>(row + k) = v[i];
    }
    sum(v[i], k);
  }
  auto rest = [&](auto step) {
    if constexpr (NV == 8)
      for (int k = (tid + NV * 256) * 4; k < ld; k += 1024) step(k);
  };
  rest([&](int k) {
    f32x4 a = *reinterpret_cast<const f32x4*>(row + k);
    if (add) {
      const V4<T> more = *reinterpret_cast<const V4<T>*>(add + (int64_t)t * ld_add + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] += (float)more[e];
      *reinterpret_cast<f32x4*>(row + k) = a;
    }
    sum(a, k);
  });
  if (!out) return;
  float mean = 0.f;
  if (!rms) {
    s = wave_sum(s);
    if (lane == 0) part[0][wave] = s;
    __syncthreads();
    mean = (part[0][0] + part[0][1] + part[0][2] + part[0][3]) / (float)n;
  }
  float q = 0.f;
  auto dev2 = [&](const f32x4& a, int k) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float c = k + e < n ? a[e] - mean : 0.f;
      q = fmaf(c, c, q);
    }
  };
#pragma unroll
  for (int i = 0; i < NV; ++i) dev2(v[i], (tid + i * 256) * 4);
  rest([&](int k) { dev2(*reinterpret_cast<const f32x4*>(row + k), k); });
  q = wave_sum(q);
  if (lane == 0) part[1][wave] = q;
  __syncthreads();
  const float rstd = 1.f / sqrtf((part[1][0] + part[1][1] + part[1][2] + part[1][3]) / (float)n + eps);
  auto put = [&](const f32x4& a, const f32x4& g, int k) {
    V4<T> o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (T)((a[e] - mean) * rstd * g[e]);
    *reinterpret_cast<V4<T>*>(out + (int64_t)t * ld + k) = o;
  };
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = (tid + i * 256) * 4;
    if (k < ld) put(v[i], w[i], k);
  }
  rest([&](int k) { put(*reinterpret_cast<const f32x4*>(row + k), *reinterpret_cast<const f32x4*>(norm_w + k), k); });
}

template <typename T>
static void launch_add_norm(int M, hipStream_t st, float* x, int64_t ldx, const int* rows, const T* add, int64_t ld_add, const float* norm_w, T* out, int n, int ld, float eps, int rms) {
  auto* fn = ld <= 1024 ? add_norm_kernel<T, 1> : ld <= 2048 ? add_norm_kernel<T, 2> : ld <= 4096 ? add_norm_kernel<T, 4> : add_norm_kernel<T, 8>;
  hipLaunchKernelGGL(fn, dim3(M), dim3(256), 0, st, x, ldx, rows, add, ld_add, norm_w, out, n, ld, eps, rms);
}

// x += scale (rms norm of a + rms norm of b) + add; one workgroup per row.  NV times 1024 columns are asked for at once, all that is read of them; NV = 0: any number, read as they come
template <typename T, int NV>
__global__ __launch_bounds__(256) void merge_kernel(float* x, const T* a, int64_t ld_a, const T* b, int64_t ld_b, const T* add,
                                                    int64_t ld_add, const float* wa, const float* wb, int n, int ld, float eps,
                                                    float scale) {
  __shared__ float part[2][4];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  a += (int64_t)t * ld_a;
  b += (int64_t)t * ld_b;
  float* row = x + (int64_t)t * ld;
  float sa = 0.f, sb = 0.f;
  struct Four {
    V4<T> a, b, d;
    f32x4 x, wa, wb;
  };
  auto squares = [&](const Four& u) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sa = fmaf((float)u.a[e], (float)u.a[e], sa);
      sb = fmaf((float)u.b[e], (float)u.b[e], sb);
    }
  };
  auto branches = [&](Four& u, int k) {
    u.a = *reinterpret_cast<const V4<T>*>(a + k);
    u.b = *reinterpret_cast<const V4<T>*>(b + k);
  };
  auto others = [&](Four& u, int k) {
    u.wa = *reinterpret_cast<const f32x4*>(wa + k);
    u.wb = *reinterpret_cast<const f32x4*>(wb + k);
    u.x = *reinterpret_cast<const f32x4*>(row + k);
    if (add) u.d = *reinterpret_cast<const V4<T>*>(add + (int64_t)t * ld_add + k);
  };
  [[maybe_unused]] Four held[NV ? NV : 1];
  if constexpr (NV > 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) branches(held[i], min((tid + 256 * i) * 4, ld - 4));
#pragma unroll
    for (int i = 0; i < NV; ++i) others(held[i], min((tid + 256 * i) * 4, ld - 4));
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if ((tid + 256 * i) * 4 < ld) squares(held[i]);   // (padding columns are zeros)
  } else {
    for (int k = tid * 4; k < ld; k += 1024) {
      Four u;
      branches(u, k);
      squares(u);
    }
  }
  sa = wave_sum(sa);
  sb = wave_sum(sb);
  if (lane == 0) part[0][wave] = sa, part[1][wave] = sb;
  __syncthreads();
  const float ra = scale / sqrtf((part[0][0] + part[0][1] + part[0][2] + part[0][3]) / (float)n + eps);
  const float rb = scale / sqrtf((part[1][0] + part[1][1] + part[1][2] + part[1][3]) / (float)n + eps);
  auto put = [&](Four& u, int k) {
    if (add) {
#pragma unroll
      for (int e = 0; e < 4; ++e) u.x[e] += (float)u.d[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) u.x[e] += (float)u.a[e] * ra * u.wa[e] + (float)u.b[e] * rb * u.wb[e];
    *reinterpret_cast<f32x4*>(row + k) = u.x;
  };
  if constexpr (NV > 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if ((tid + 256 * i) * 4 < ld) put(held[i], (tid + 256 * i) * 4);
  } else {
    for (int k = tid * 4; k < ld; k += 1024) {
      Four u;
      branches(u, k), others(u, k);
      put(u, k);
    }
  }
}

// out [T, 2 n] = (x | x2) in the element type
template <typename T>
__global__ __launch_bounds__(256) void concat_kernel(const float* __restrict__ x, const float* __restrict__ x2, T* __restrict__ out, int n) {
  const int t = blockIdx.y, j = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (j >= 2 * n) return;
  *reinterpret_cast<V8<T>*>(out + (int64_t)t * 2 * n + j) = from_f32<T>(load8((j < n ? x + j : x2 + j - n) + (int64_t)t * n));
}

template <typename T>
__global__ __launch_bounds__(256) void glu_kernel(const T* __restrict__ in, int64_t ld_in, T* __restrict__ out, int64_t ld_out, int n,
                                                  float limit, float alpha, float up) {
  const int t = blockIdx.y, j = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (j >= n) return;
  const V8<T> v = load8(in + (int64_t)t * ld_in + 2 * j);
  V4<T> o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (T)glu((float)v[2 * e], (float)v[2 * e + 1], limit, alpha, up);
  *reinterpret_cast<V4<T>*>(out + (int64_t)t * ld_out + j) = o;
}

__global__ __launch_bounds__(1024) void argmax_kernel(const float* __restrict__ logits, int64_t ld, int V, int64_t* __restrict__ out) {
  __shared__ float sb[16];
  __shared__ int si[16];
  const float* row = logits + (int64_t)blockIdx.x * ld;
  float best = -INFINITY;
  int at = 0x7fffffff;
  auto take = [&](float v, int i) {
    if (v > best || (v == best && i < at)) {
      best = v;
      at = i;
    }
  };
  for (int i = threadIdx.x; i < V; i += 1024) take(row[i], i);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(at, o, 64);
    take(ob, oi);
  }
  if ((threadIdx.x & 63) == 0) {
    sb[threadIdx.x >> 6] = best;
    si[threadIdx.x >> 6] = at;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) take(sb[w], si[w]);
    out[blockIdx.x] = at == 0x7fffffff ? 0 : at;
  }
}

int check_linear(const vmi_hy_linear_args* a, const char* who) {
  if (!a || !a->x || !a->w || !a->y || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->groups <= 0 || a->dtype < 0 || a->dtype > 1 ||
      (a->x_kind == VMI_HY_X_NORM && (!a->norm_w || a->norm_n <= 0 || a->norm_n > a->K)) || (a->x_kind == VMI_HY_X_CONCAT && !a->x2) ||
      (a->epilogue == VMI_HY_E_GATED && !a->gate) || (a->epilogue == VMI_HY_E_STORE_GLU && !a->y2))
    return fail(VMI_HY_E_ARG, who, "null pointer, non-positive size or unknown element type");
  if ((a->K & 31) || (a->N & 15) || (a->x_kind == VMI_HY_X_CONCAT && (a->K & 63)) || (a->ldx & 7) || (a->x_gstride & 7) ||
      (a->epilogue != VMI_HY_E_FLOAT && ((a->ldy & 3) || (a->y_gstride & 3))) || ((uintptr_t)a->x & 15) || ((uintptr_t)a->w & 15) ||
      ((uintptr_t)a->y & 15) || ((uintptr_t)a->normed & 15) ||
      (a->epilogue == VMI_HY_E_FLOAT && (a->n_out <= 0 || a->n_out > a->N || a->groups != 1)) ||
      (a->epilogue == VMI_HY_E_STORE_GLU && (a->n_split < 0 || a->n_split > a->N || (a->n_split & 15) || (a->ldy2 & 1) ||
                                             ((uintptr_t)a->y2 & 7) || a->groups != 1)))
    return fail(VMI_HY_E_SHAPE, who, "needs K % 32 == 0, N % 16 == 0 and 16-byte aligned rows");
  return VMI_HY_OK;
}

}  // namespace vmi_hybrid

using namespace vmi_hybrid;

extern "C" {

int32_t vmi_hy_linear_normed(int32_t M, int32_t N, int32_t K, int32_t groups, int32_t dtype) {
  return dtype == VMI_HY_BF16 && M > 0 && N > 0 && K > 0 && groups == 1 && (norm_first(M, N, K) || (K < 4096 && held_rows_pay(M, N, K, false)));
}

int32_t vmi_hy_linear_resident(int32_t M, int32_t N, int32_t K, int32_t dtype) {
  return dtype == VMI_HY_BF16 && M > 0 && N > 0 && K > 0 && resident_kind(M, N, K) != 0;
}

int32_t vmi_hy_linear_slabs(int32_t M, int32_t N, int32_t K, int32_t dtype) {
  return dtype == VMI_HY_BF16 && M > 0 && N > 0 && K > 0 && (K & 31) == 0 && (N & 15) == 0 ? norm_slabs(M, N, K) : 0;
}

int32_t vmi_hy_linear_plain(int32_t M, int32_t N, int32_t K, int32_t groups, int32_t dtype) {
  return dtype == VMI_HY_BF16 && M > 0 && N > 0 && K > 0 && groups > 0 && plain_rows_fit(M, N, K, groups);
}

int32_t vmi_hy_linear_held(int32_t M, int32_t N, int32_t K, int32_t dtype) {
  return K < 4096 && vmi_hy_linear_holds(M, N, K, 0, dtype);
}

int32_t vmi_hy_linear_holds(int32_t M, int32_t N, int32_t K, int32_t stored, int32_t dtype) {
  return dtype == VMI_HY_BF16 && M > 0 && N > 0 && K > 0 && held_rows_pay(M, N, K, stored != 0);
}

int vmi_hy_linear(const vmi_hy_linear_args* a, void* stream) {
  static const char* who = "vmi_hy_linear";
  if (int rc = check_linear(a, who)) return rc;
  DeviceScope dev(a->device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (a->x_kind == VMI_HY_X_NORM && a->normed && a->dtype == VMI_HY_BF16 && a->epilogue != VMI_HY_E_RESIDUAL && a->epilogue != VMI_HY_E_GATED) {
    if (launch_norm_few(*a, st) != VMI_HY_OK)
      launch_add_norm<b16>(a->M, st, const_cast<float*>(static_cast<const float*>(a->x)), a->ldx, a->rows, nullptr, (int64_t)0, a->norm_w, static_cast<b16*>(a->normed), a->norm_n, a->K, a->eps, a->rms);
    vmi_hy_linear_args rows = *a;
    rows.x = a->normed, rows.ldx = a->K, rows.x_gstride = 0, rows.rows = nullptr, rows.x_kind = VMI_HY_X_ROWS;   // (all groups read the same rows)
    return linear_normed(rows, st);
  }
  return a->dtype == VMI_HY_BF16 ? linear_kind<b16>(*a, st) : linear_kind<float>(*a, st);
}

int vmi_hy_step_inputs(const void* host, void* dev_to, int64_t bytes, const int64_t* ids, int64_t* ids_out, int32_t n, int32_t device, void* stream) {
  static const char* who = "vmi_hy_step_inputs";
  const vmi_step::Inputs p{static_cast<const char*>(host), static_cast<char*>(dev_to), bytes, 0, 0, 0, n, ids, ids_out};
  if (!vmi_step::inputs_fit(p)) return fail(VMI_HY_E_ARG, who, "null pointer, a size out of range, or memory that is not aligned to 16 bytes");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  vmi_step::launch_inputs(p, static_cast<hipStream_t>(stream));
  return launched(who);
}

int vmi_hy_embed(const int64_t* ids, const void* table, float* x, int32_t T, int32_t width, int32_t ld, int32_t vocab, float scale,
                 int32_t device, void* stream) {
  static const char* who = "vmi_hy_embed";
  if (!ids || !table || !x || T <= 0 || width <= 0 || ld < width || (ld & 3) || vocab <= 0) return fail(VMI_HY_E_ARG, who, "bad argument");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipLaunchKernelGGL(embed_kernel, dim3(T), dim3(256), 0, static_cast<hipStream_t>(stream), ids, static_cast<const b16*>(table), x,
                     width, ld, vocab, scale);
  return launched(who);
}

int vmi_hy_add_norm(float* x, const void* add, int64_t ld_add, const float* norm_w, void* out, int32_t T, int32_t n, int32_t ld,
                    float eps, int32_t rms, int32_t dtype, int32_t device, void* stream) {
  static const char* who = "vmi_hy_add_norm";
  if (!x || T <= 0 || n <= 0 || ld < n || (ld & 3) || (add && (ld_add & 3)) || (out && !norm_w)) return fail(VMI_HY_E_ARG, who, "bad argument");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == VMI_HY_BF16)
    launch_add_norm<b16>(T, st, x, (int64_t)ld, nullptr, static_cast<const b16*>(add), ld_add, norm_w,
                       static_cast<b16*>(out), n, ld, eps, rms);
  else
    launch_add_norm<float>(T, st, x, (int64_t)ld, nullptr, static_cast<const float*>(add), ld_add, norm_w,
                       static_cast<float*>(out), n, ld, eps, rms);
  return launched(who);
}

int vmi_hy_glu(const void* in, int64_t ld_in, void* out, int64_t ld_out, int32_t T, int32_t n, float limit, float alpha,
               float up, int32_t dtype, int32_t device, void* stream) {
  static const char* who = "vmi_hy_glu";
  if (!in || !out || T <= 0 || T > 65535 || n <= 0 || (n & 3) || (ld_in & 7) || (ld_out & 3)) return fail(VMI_HY_E_ARG, who, "bad argument");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((n / 4 + 255) / 256, T);
  if (dtype == VMI_HY_BF16)
    hipLaunchKernelGGL(glu_kernel<b16>, grid, dim3(256), 0, st, static_cast<const b16*>(in), ld_in, static_cast<b16*>(out), ld_out, n,
                       limit, alpha, up);
  else
    hipLaunchKernelGGL(glu_kernel<float>, grid, dim3(256), 0, st, static_cast<const float*>(in), ld_in, static_cast<float*>(out), ld_out, n,
                       limit, alpha, up);
  return launched(who);
}

int vmi_hy_merge(float* x, const void* a, int64_t ld_a, const void* b, int64_t ld_b, const void* add, int64_t ld_add, const float* wa,
                 const float* wb, int32_t T, int32_t n, int32_t ld, float eps, float scale, int32_t dtype, int32_t device,
                 void* stream) {
  static const char* who = "vmi_hy_merge";
  if (!x || !a || !b || !wa || !wb || T <= 0 || n <= 0 || ld < n || (ld & 3) || (ld_a & 3) || (ld_b & 3) || (add && (ld_add & 3)))
    return fail(VMI_HY_E_ARG, who, "bad argument");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto go = [&](auto kind) {
    using T_ = decltype(kind);
    auto* fn = ld <= 1024 ? merge_kernel<T_, 1> : ld <= 2048 ? merge_kernel<T_, 2> : ld <= 4096 ? merge_kernel<T_, 4> : merge_kernel<T_, 0>;
    hipLaunchKernelGGL(fn, dim3(T), dim3(256), 0, st, x, static_cast<const T_*>(a), ld_a, static_cast<const T_*>(b), ld_b, static_cast<const T_*>(add), ld_add, wa, wb, n, ld, eps, scale);
  };
  if (dtype == VMI_HY_BF16) go(b16{});
  else go(float{});
  return launched(who);
}

int vmi_hy_concat(const float* x, const float* x2, void* out, int32_t T, int32_t n, int32_t dtype, int32_t device, void* stream) {
  static const char* who = "vmi_hy_concat";
  if (!x || !x2 || !out || T <= 0 || T > 65535 || n <= 0 || (n & 7)) return fail(VMI_HY_E_ARG, who, "bad argument");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((2 * n / 8 + 255) / 256, T);
  if (dtype == VMI_HY_BF16)
    hipLaunchKernelGGL(concat_kernel<b16>, grid, dim3(256), 0, st, x, x2, static_cast<b16*>(out), n);
  else
    hipLaunchKernelGGL(concat_kernel<float>, grid, dim3(256), 0, st, x, x2, static_cast<float*>(out), n);
  return launched(who);
}

int vmi_hy_argmax(const float* logits, int64_t ld, int32_t rows, int32_t V, int64_t* out, int32_t device, void* stream) {
  static const char* who = "vmi_hy_argmax";
  if (!logits || !out || rows <= 0 || V <= 0 || ld < V) return fail(VMI_HY_E_ARG, who, "bad argument");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipLaunchKernelGGL(argmax_kernel, dim3(rows), dim3(1024), 0, static_cast<hipStream_t>(stream), logits, ld, V, out);
  return launched(who);
}

const char* vmi_hybrid_last_error(void) { return g_err.c_str(); }
int32_t vmi_hybrid_abi_version(void) { return VMI_HYBRID_ABI_VERSION; }
const char* vmi_hybrid_target_arch(void) { return "gfx950"; }

}  // extern "C"
