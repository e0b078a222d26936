// Causal attention over whole prompts, and their keys and values into the paged cache, in one launch per layer (included by
// gpt2_layer.hip; include/vmi_gpt2_layer.h: vmi_gpt2_prompt_attention_f16).
//
// A prompt's q, k and v lie in the projection's rows, so nothing is read back from the cache: a workgroup takes 64 * MI query
// positions of one head and walks the keys up to its last position in tiles of 64, each through LDS once (requested one tile ahead,
// two buffers, one barrier a tile).  A wave owns 16 * MI queries for all of it:
//   * scores are formed transposed, S^T = K Q^T (D[row = key 4 kc + r][col = query r16]), so a lane keeps the scores of ONE query: its
//     statistics need no LDS, its maximum two cross-lane swaps, its sum a product with ones, and its probabilities, as they lie, are the B operand of
//     O^T = V^T P^T: the sum over keys may take them in any order, so k-index 8 kc + e of a step of 32 stands for key 4 kc + e
//     (e < 4) and 16 + 4 kc + e - 4, and the V^T operand is read column-wise from LDS in that same order (ds_read_b64_tr_b16);
//   * the key tiles that lie on the workgroup's own positions are its prompt's pages: they leave from LDS as whole 16-byte pieces of
//     the cache's layout, K[blk, h, d / 8, off, d % 8] and V[blk, h, d, off] — the bytes that reshape_and_cache would write.
// Scores, softmax and accumulators are fp32; a probability is rounded once to half and what is summed is what multiplies V.
//
// What bounds it: the vector unit's share of the softmax (a maximum, a multiply-add, an exponential and half a conversion a score; the scale is in the multiply-add, the sums are
// in the matrix cores, which are mostly idle) and the chain of a tile (LDS, scores, softmax, values: 0.65 us) times the longest prompt's tiles.  So the longest walks begin first,
// over all heads: as one head behind the other the last head's began when the first ones' were done.  Keys shared out over two or four groups of waves of a workgroup, their sums
// merged at the end: one of 900 13.3 -> 12.3 us, 6 of 900 17.2 -> 15.5, but 24 of up to 512 17.7 -> 21.5 and up to 200 tokens behind everywhere: not kept.
// As a sequence of its own per position, for paged_attention_v1, every position read its keys again, and the cache was written by a launch in front in 2-byte pieces.
// 24 prompts of up to 512 tokens (6 439 in all), 12 heads of 64, a layer: 205.6 + 30.2 -> 23.2 us, with a scaled, rounded and added score and heads outermost -> 17.7; one
// prompt of 37: 5.1 + 3.2 -> 3.9 us, of 900 16.8 -> 13.3; 16 heads of 128, 4 of 900 34.2 -> 27.1.
#pragma once
#include "mfma_tiles.hpp"

namespace vmi_layer {

struct PromptParams {
  const h16* qkv;         // [T][ld]: q | k | v, heads * D columns each
  int64_t ld;
  h16* out;               // [T][ldo]
  int64_t ldo;
  const int32_t* tiles;   // [n][4]: prompt, its first packed row, the tile's first position, the prompt's length
  const int32_t* table;   // [prompts][table_ld]: this layer's blocks
  int table_ld, heads;
  h16* kcache;
  h16* vcache;
  int64_t bstride, hstride;
  float scale2;           // scale * log2(e): scores in units of log 2
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// four consecutive rows of one column of an LDS tile: lane r16 of each 16 holds column col0 + r16
__device__ __forceinline__ h16x4 column4(const h16* tile, int ld, int row0, int col0, int r16) {
  const h16* a = tile + (row0 + (r16 >> 2)) * ld + col0 + 4 * (r16 & 3);
  return __builtin_bit_cast(h16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)a));
}
__device__ __forceinline__ h16x8 join(const h16x4& lo, const h16x4& hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }

// over the four lanes that share r16: the rows of 16 lanes are swapped pairwise, no LDS round trip
template <typename F>
__device__ __forceinline__ float over_kc(float v, F op) {
  const uint32_t a = __builtin_bit_cast(uint32_t, v);
  const auto s = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  const uint32_t b = __builtin_bit_cast(uint32_t, op(__builtin_bit_cast(float, (uint32_t)s[0]), __builtin_bit_cast(float, (uint32_t)s[1])));
  const auto t = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return op(__builtin_bit_cast(float, (uint32_t)t[0]), __builtin_bit_cast(float, (uint32_t)t[1]));
}

constexpr int PKT = 64;      // keys of a tile: four pages of 16
constexpr int PROMPT_BS = 16;

// One query row by one wave over keys 0 .. q, with nothing but those in any sum: lanes share the keys for the scores and the columns for the values.  k: key
// 0 of the head, its value E further on; kept for rows whose sums are NaN otherwise
template <int D>
__device__ void one_query(const h16* qrow, const h16* k, int64_t ld, int q, float scale2, h16* out, int E, int lane) {
  auto score = [&](int key) {
    float s = 0.f;
    for (int d = 0; d < D; d += 8) {
      const h16x8 a = *reinterpret_cast<const h16x8*>(qrow + d), b = *reinterpret_cast<const h16x8*>(k + key * ld + d);
#pragma unroll
      for (int e = 0; e < 8; ++e) s = fmaf((float)a[e], (float)b[e], s);
    }
    return s * scale2;
  };
  float mx = -1e30f;
  for (int key = lane; key <= q; key += 64) mx = fmaxf(mx, score(key));
#pragma unroll
  for (int i = 1; i < 64; i <<= 1) mx = fmaxf(mx, __shfl_xor(mx, i, 64));
  float sum = 0.f, o[D / 64];
#pragma unroll
  for (int i = 0; i < D / 64; ++i) o[i] = 0.f;
  for (int key0 = 0; key0 <= q; key0 += 64) {
    const int n = min(64, q + 1 - key0);
    const float pr = lane < n ? (float)(h16)__builtin_amdgcn_exp2f(score(key0 + lane) - mx) : 0.f;
    sum += pr;
    for (int j = 0; j < n; ++j) {
      const float pj = __shfl(pr, j, 64);
#pragma unroll
      for (int i = 0; i < D / 64; ++i) o[i] = fmaf(pj, (float)k[(key0 + j) * ld + E + lane + 64 * i], o[i]);
    }
  }
#pragma unroll
  for (int i = 1; i < 64; i <<= 1) sum += __shfl_xor(sum, i, 64);
#pragma unroll
  for (int i = 0; i < D / 64; ++i) out[lane + 64 * i] = (h16)(o[i] / sum);
}

template <int D, int MI>
__global__ __launch_bounds__(256, 2) void prompt_attention_kernel(const PromptParams p) {
  constexpr int LD = D + 8, NK = D / 32, NT = D / 16, UPR = D / 8, U = PKT * UPR / 256;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  h16* lds = reinterpret_cast<h16*>(smem);   // [2 buffers][K, V][64][LD]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kc = lane >> 4, r16 = lane & 15;
  const int h = blockIdx.x % p.heads;   // (the heads of a tile one behind the other: the longest walks, which the list has first, all begin first)
  const int4 tile = *reinterpret_cast<const int4*>(p.tiles + 4 * (blockIdx.x / p.heads));
  const int q0 = tile.z, len = tile.w, E = p.heads * D;
  const h16* row0 = p.qkv + (int64_t)tile.y * p.ld + h * D;
  const int32_t* table = p.table + (int64_t)tile.x * p.table_ld;
  const int end = min(len, q0 + 64 * MI), nkt = (end + PKT - 1) / PKT;

  h16x8 kr[U], vr[U];
  auto load = [&](int kt) {   // (keys past the end repeat the last one: no lane-wise condition around a load)
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = tid + 256 * i;
      const h16* src = row0 + (int64_t)min(kt * PKT + u / UPR, len - 1) * p.ld + E + (u % UPR) * 8;
      kr[i] = *reinterpret_cast<const h16x8*>(src);
      vr[i] = *reinterpret_cast<const h16x8*>(src + E);
    }
  };
  load(0);
  // the pages of the workgroup's own positions, asked for now: behind its last tile each of them was a trip to memory that nothing else was left to hide
  int page[MI][U];
#pragma unroll
  for (int m = 0; m < MI; ++m)
#pragma unroll
    for (int i = 0; i < U; ++i) page[m][i] = table[min(q0 + m * PKT + (tid + 256 * i) / (16 * UPR) * PROMPT_BS, len - 1) / PROMPT_BS];
  const int w0 = q0 + wave * 16 * MI;   // this wave's first position
  h16x8 qf[MI][NK];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int k = 0; k < NK; ++k)
      qf[mi][k] = *reinterpret_cast<const h16x8*>(row0 + (int64_t)min(w0 + mi * 16 + r16, len - 1) * p.ld + 32 * k + 8 * kc);
  h16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (h16)1.f;
  f32x4 o[MI][NT];
  float mrun[MI], lrun[MI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    mrun[mi] = -1e30f;
    lrun[mi] = 0.f;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) o[mi][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  for (int kt = 0; kt < nkt; ++kt) {
    h16* ks = lds + (kt & 1) * 2 * PKT * LD;
    h16* vs = ks + PKT * LD;
    const int key0 = kt * PKT;
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = tid + 256 * i;
      *reinterpret_cast<h16x8*>(ks + (u / UPR) * LD + (u % UPR) * 8) = kr[i];
      *reinterpret_cast<h16x8*>(vs + (u / UPR) * LD + (u % UPR) * 8) = vr[i];
    }
    if (kt + 1 < nkt) load(kt + 1);
    __syncthreads();   // (the writes of tile kt + 1 go where tile kt - 1 was read, which every wave has left behind)
    if (key0 >= q0) {   // this workgroup's own positions: four pages into the cache
      int64_t at_page[U];
#pragma unroll
      for (int i = 0; i < U; ++i) at_page[i] = (MI > 1 && key0 > q0 ? page[MI - 1][i] : page[0][i]) * p.bstride + h * p.hstride;
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int u = tid + 256 * i, pg = u / (16 * UPR), off = u & 15, d8 = (u >> 4) % UPR, pos = key0 + pg * PROMPT_BS;
        if (pos + off < len)
          *reinterpret_cast<h16x8*>(p.kcache + at_page[i] + (d8 * PROMPT_BS + off) * 8) =
              *reinterpret_cast<const h16x8*>(ks + (pg * PROMPT_BS + off) * LD + d8 * 8);
      }
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int g = (tid >> 4) + 16 * i, half = g & 1, nt = (g >> 1) % NT, pg = g / (2 * NT), pos = key0 + pg * PROMPT_BS + half * 8;
        const int at = pg * PROMPT_BS + half * 8;
        const h16x8 v = join(column4(vs, LD, at, nt * 16, r16), column4(vs, LD, at + 4, nt * 16, r16));
        if (pos < len) {
          h16* dst = p.vcache + at_page[i] + (nt * 16 + r16) * PROMPT_BS + half * 8;
          if (pos + 8 <= len) {
            *reinterpret_cast<h16x8*>(dst) = v;
          } else {   // the prompt ends inside: slots behind it are not this prompt's to write
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (pos + e < len) dst[e] = v[e];
          }
        }
      }
    }
    if (w0 >= len || key0 > w0 + 16 * MI - 1) continue;   // (wave-uniform: none of its queries exists, or sees the tile)
    f32x4 sc[MI][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) sc[mi][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const h16x8 kf = *reinterpret_cast<const h16x8*>(ks + (j * 16 + r16) * LD + 32 * k + 8 * kc);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) sc[mi][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[mi][k], sc[mi][j], 0, 0, 0);
      }
    }
    const bool whole = key0 + PKT - 1 <= w0;   // every query sees every key
    if (!whole) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (key0 + j * 16 + 4 * kc + r > w0 + mi * 16 + r16) sc[mi][j][r] = -INFINITY;
    }
    h16x8 pf[MI][2];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      float mx = sc[mi][0][0];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[mi][j][r]);
      mx = fmaxf(mrun[mi], p.scale2 * over_kc(mx, [](float a, float b) { return fmaxf(a, b); }));
      const float alpha = __builtin_amdgcn_exp2f(mrun[mi] - mx);
      mrun[mi] = mx;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) pf[mi][j >> 1][(j & 1) * 4 + r] = (h16)__builtin_amdgcn_exp2f(__builtin_fmaf(sc[mi][j][r], p.scale2, -mx));
      // (what is summed is what multiplies V: a product with ones, whose every row is the sums)
      f32x4 sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2; ++k) sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pf[mi][k], sum, 0, 0, 0);
      lrun[mi] = __builtin_fmaf(lrun[mi], alpha, sum[0]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) o[mi][nt] *= alpha;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const h16x8 vf = join(column4(vs, LD, 32 * k + 4 * kc, nt * 16, r16), column4(vs, LD, 32 * k + 16 + 4 * kc, nt * 16, r16));
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) o[mi][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf[mi][k], o[mi][nt], 0, 0, 0);
      }
  }
  // A key that a query does not see has a probability of 0, which times an infinite or NaN value is NaN in the matrix cores: a wave whose sums hold a NaN
  // does its rows again, one by one, and leaves out what is masked.  (One add and compare a value, once: 24 prompts of up to 512 tokens as before)
  float any = 0.f;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) any += (o[mi][nt][0] + o[mi][nt][1]) + (o[mi][nt][2] + o[mi][nt][3]);
  if (__ballot(any != any) != 0) {
    const int last = min(w0 + 16 * MI, len);
    for (int q = w0; q < last; ++q) one_query<D>(row0 + (int64_t)q * p.ld, row0 + E, p.ld, q, p.scale2, p.out + (int64_t)(tile.y + q) * p.ldo + h * D, E, lane);
    return;
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const float inv = 1.f / lrun[mi];
    const int q = w0 + mi * 16 + r16;
    if (q >= len) continue;
    h16* out = p.out + (int64_t)(tile.y + q) * p.ldo + h * D + 4 * kc;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      h16x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = (h16)(o[mi][nt][r] * inv);
      *reinterpret_cast<h16x4*>(out + nt * 16) = y;
    }
  }
}

// x += add (if given), and the layer norm of x (of `rows` of it) in half: one wave a row, the row in registers between the sum, the two
// passes of its statistics (fp32) and the result.  Bound by memory: two rows read, two written.  As torch's add and layer_norm, two
// launches that between them read the stream three times, 6 439 rows of 768: 6.0 + 13.5 -> 9.1 us.
template <int UPL>   // 16-byte units of a row per lane
__global__ __launch_bounds__(256) void add_norm_kernel(h16* __restrict__ x, const h16* __restrict__ add, const int32_t* __restrict__ rows,
                                                       const h16* __restrict__ gamma, const h16* __restrict__ beta, h16* __restrict__ out,
                                                       int M, int E, float eps) {
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, units = E >> 3;
  if (m >= M) return;
  h16* row = x + (int64_t)(rows ? rows[m] : m) * E;
  h16x8 v[UPL], y[UPL];
  float f[UPL][8];
#pragma unroll
  for (int i = 0; i < UPL; ++i) {   // (lanes past the row read its last unit again)
    const int u = min(lane + 64 * i, units - 1) * 8;
    v[i] = *reinterpret_cast<const h16x8*>(row + u);
    if (add) y[i] = *reinterpret_cast<const h16x8*>(add + (int64_t)m * E + u);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    const bool on = lane + 64 * i < units;
    if (add) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] = (h16)((float)v[i][e] + (float)y[i][e]);
      if (on) *reinterpret_cast<h16x8*>(row + (lane + 64 * i) * 8) = v[i];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      f[i][e] = (float)v[i][e];
      s += on ? f[i][e] : 0.f;
    }
  }
  const float mean = group_sum<64>(s) / (float)E;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    const bool on = lane + 64 * i < units;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      f[i][e] -= mean;
      q = on ? fmaf(f[i][e], f[i][e], q) : q;
    }
  }
  const float rstd = rsqrtf(group_sum<64>(q) / (float)E + eps);
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    if (lane + 64 * i >= units) continue;
    const int u = (lane + 64 * i) * 8;
    const h16x8 g = *reinterpret_cast<const h16x8*>(gamma + u), b = *reinterpret_cast<const h16x8*>(beta + u);
    h16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (h16)fmaf(f[i][e] * rstd, (float)g[e], (float)b[e]);
    *reinterpret_cast<h16x8*>(out + (int64_t)m * E + u) = o;
  }
}

// Linear layers of many rows, packed weights (mfma_tiles.hpp): bias and GELU on what a lane holds, the residual add on its share of the lines that leave, the rounding points of
// the few-row kernels.  The bias is asked for at the start, residuals too where a tile leaves the registers for it, else when the product is done.
template <int MI, int NI, int D, int EPI>
__global__ __launch_bounds__(256, 2) void tiles_kernel(const LinearParams p) {
  constexpr bool ADD = EPI == VMI_LAYER_EPI_BIAS_RESIDUAL, EARLY = MI * NI <= 12, EARLY_BIAS = MI * NI <= 24;
  constexpr int PIECES = 8 * NI, MINE = MI / 2 * NI;   // sixteen bytes of results: of a row, and those of a lane
  h16x4 bias[NI];
  h16x8 res[ADD ? MINE : 1];
  typedef h16x8 Eight __attribute__((aligned(8)));   // (rows of four are all that is asked of a residual: one request all the same)
  const bool wide = ((p.ldy & 7) | ((uintptr_t)p.y & 15)) == 0;
  auto ask_bias = [&](const vmi_tiles::Where& at) {
#pragma unroll
    for (int n = 0; n < NI; ++n) bias[n] = Tail::load_bias(p, min(at.s0 + at.wave * NI + n, at.SL - 1) * 16 + 4 * at.kc);
  };
  auto ask = [&](const vmi_tiles::Where& at) {   // (in the order of vmi_tiles::lines_out; rows and columns past the last: those again)
#pragma unroll
    for (int k = 0; k < MINE; ++k) {
      const int u = (int)threadIdx.x + 256 * (k % NI), row = u / PIECES, piece = u - row * PIECES;
      const h16* from = p.res + (int64_t)min(at.m0 + 32 * (k / NI) + row, p.M - 1) * p.ldr + min(at.s0 * 16 + 8 * piece, p.N - 8);
      res[k] = *reinterpret_cast<const Eight*>(from);
    }
  };
  vmi_tiles::tiles_product<vmi_tiles::Half, MI, NI, D>(
      p.x, p.ldx, p.w, p.M, p.N, p.K,
      [&](const vmi_tiles::Where& at) {
        if constexpr (EARLY_BIAS) ask_bias(at);
        if constexpr (ADD && EARLY) ask(at);
      },
      [&](const f32x4(&acc)[NI][MI], const vmi_tiles::Where& at) {
        if constexpr (ADD && !EARLY) ask(at);
        if constexpr (!EARLY_BIAS) ask_bias(at);
        auto pack = [&](int n, int i) {
          h16x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o[r] = (h16)(acc[n][i][r] + (float)bias[n][r]);   // the linear layer's own half output
            if constexpr (EPI == VMI_LAYER_EPI_BIAS_GELU) o[r] = (h16)gelu((float)o[r]);
          }
          return __builtin_bit_cast(vmi_tiles::u32x2, o);
        };
        auto put = [&](int row, int piece, vmi_tiles::u32x4 v, int k) {
          const int m = at.m0 + row, n = at.s0 * 16 + 8 * piece;
          if constexpr (ADD) {
            const h16x8 a = __builtin_bit_cast(h16x8, v);
            h16x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (h16)((float)res[k][e] + (float)a[e]);
            v = __builtin_bit_cast(vmi_tiles::u32x4, o);
          }
          vmi_tiles::put_piece(m < p.M && n < p.N, p.y + (int64_t)m * p.ldy + n, v, wide);
        };
        // (GELU takes the vector pipes as long as the product takes the matrix cores, so its waves go on one by one: 2000 rows, N 3072, K 768 15.6 us, by lines 15.9; 6400 40.6 / 44)
        if constexpr (EPI == VMI_LAYER_EPI_BIAS_GELU && NI % 2 == 0) vmi_tiles::pairs_out<MI, NI>(at, pack, put);
        else vmi_tiles::lines_out<vmi_tiles::u32x2, MI, NI, EPI == VMI_LAYER_EPI_BIAS_GELU>(at, pack, put);
      });
}

}  // namespace vmi_layer
