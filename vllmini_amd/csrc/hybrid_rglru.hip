// The recurrent block between its projections (include/vmi_hybrid.h): causal convolution -> block-diagonal gates -> gated linear
// recurrence -> product with gelu(y).
//
// The packed tokens are cut into row tiles of BM consecutive rows, whatever entries they belong to.  A workgroup takes one row
// tile x up to 64 channels of one gate block: the convolution of the block's channels goes to LDS (element type), both gate
// matrices run on the matrix cores (A = gate rows = channels, B = u rows = tokens, fp32 accumulation), and everything behind the
// product is fp32: r, i, log a = decay * r, a, b = sqrt(1 - a^2) * i * u.  A token that opens an entry's portion folds the state
// of its slot in at once (b += a * S, a = 0), so one uniform walk S = a S + b, P = a P over the tile serves any mix of entries:
// P is zero from an opening token on and the product of the decays in front of one — only the rows of a tile's LEADING segment
// (a portion that began in an earlier tile) are unfinished, by P * (the carry into the tile).  Batches whose portions all fit
// their tiles — every decode step — are one launch; otherwise a second kernel runs the carries from tile to tile and a third
// finishes the leading rows.
//
// The convolution's tail (the last taps - 1 inputs of a sequence) has two halves: a step reads half `flip` and writes the other
// one, so no workgroup can overwrite what another still reads.
#include "hybrid_common.hpp"

namespace vmi_hybrid {

constexpr int CT = 64;      // channels of a workgroup
constexpr int KCH = 256;    // channels of u in LDS at a time
constexpr int MAX_TAPS = 16;

struct RowMeta {
  int seq, qs, len, ctx, slot, flip, first, last;
};

template <typename T, int BM>
struct Lds {
  static constexpr int LDU = KCH + 16 / (int)sizeof(T), LDA = CT + 4;
  T u[BM * LDU];
  float a[BM * LDA];
  float b[BM * LDA];
  float end[2][4][CT];
  RowMeta meta[BM];
};

// convolution of 8 channels for the token of row m.  TAPS = 0: any number of taps; else exactly that many, every load issued
// without a condition around it (taps before the start read a valid row and count zero), so that all of them are in flight
template <typename T, int TAPS>
__device__ __forceinline__ f32x8 conv8(const vmi_hy_rglru_args& p, const RowMeta& r, int t, int c) {
  f32x8 acc = load8(p.conv_b + c);
  const T* in = static_cast<const T*>(p.yx) + p.width + c;
  const int taps = TAPS ? TAPS : p.taps, pos = r.ctx + t - r.qs;
  // tail entries: positions ctx - (taps - 1) .. ctx - 1
  const T* tail = static_cast<const T*>(p.tail) + ((int64_t)r.slot * 2 + r.flip) * (taps - 1) * p.width + c;
  auto tap = [&](int j) {
    const int back = taps - 1 - j;
    const T* src = t - back >= r.qs ? in + (int64_t)(t - back) * p.ldx
                   : pos >= back    ? tail + (int64_t)(pos - back - (r.ctx - (taps - 1))) * p.width
                                    : in + (int64_t)t * p.ldx;
    const V8<T> v = load8(src);
    const f32x8 w = load8(p.conv_w + (int64_t)j * p.width + c);
    const bool on = pos >= back;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = fmaf(w[e], on ? (float)v[e] : 0.f, acc[e]);
  };
  if constexpr (TAPS > 0) {
#pragma unroll
    for (int j = 0; j < TAPS; ++j) tap(j);
  } else {
    for (int j = 0; j < taps; ++j) tap(j);
  }
  return acc;
}

template <typename T>
__device__ __forceinline__ void store_out8(const vmi_hy_rglru_args& p, int t, int c, const f32x8& s, const f32x8& y) {
  f32x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = s[e] * gelu_tanh(y[e]);
  *reinterpret_cast<V8<T>*>(static_cast<T*>(p.out) + (int64_t)t * p.ldo + c) = from_f32<T>(o);
}

template <typename T, int BM, int TAPS>
__global__ __launch_bounds__(256, 2) void rglru_tile_kernel(const vmi_hy_rglru_args p, const vmi_hy_step s) {
  constexpr int MT = BM / 16;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  auto& L = *reinterpret_cast<Lds<T, BM>*>(smem);
  constexpr int LDU = Lds<T, BM>::LDU, LDA = Lds<T, BM>::LDA;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kc = lane >> 4, r16 = lane & 15;
  const int bw = p.width / p.blocks, per = (bw + CT - 1) / CT;
  const int blk = blockIdx.x / per, cin = (blockIdx.x % per) * CT;   // gate block, first channel inside it
  const int t0 = blockIdx.y * BM, rows = min(BM, s.T - t0);
  const int nch = min(CT, bw - cin), c0 = blk * bw + cin;            // channels of this workgroup (a multiple of 32)

  if (tid < BM) {
    RowMeta r{-1, 0, 0, 0, 0, 0, 0, 0};
    if (tid < rows) r.seq = s.tok_seq[t0 + tid];
    if (r.seq >= 0) {
      r.qs = s.q_start[r.seq];
      r.len = s.q_len[r.seq];
      r.ctx = s.ctx[r.seq];
      r.slot = s.state_slot[r.seq];
      r.flip = s.flip[r.seq];
      r.first = t0 + tid == r.qs;
      r.last = t0 + tid == r.qs + r.len - 1;
    }
    L.meta[tid] = r;
  }

  // gate products over the block's channels, KCH of them in LDS at a time
  f32x4 ar[MT], ai[MT];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) ar[mi] = ai[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool wvalid = wave * 16 < nch;
  const int64_t gsz = (int64_t)bw * bw, nks = bw >> 5;
  const T* wr = static_cast<const T*>(p.gates) + blk * gsz + ((int64_t)((cin >> 4) + wave) * nks * 64 + lane) * 8;
  const T* wi = wr + p.blocks * gsz;
  // requested now, used behind the products
  const int cl = wave * 16 + 4 * kc;
  f32x4 br, bi, dec, S0[MT];
  if (wvalid) {
    br = *reinterpret_cast<const f32x4*>(p.gate_b + c0 + cl);
    bi = *reinterpret_cast<const f32x4*>(p.gate_b + p.width + c0 + cl);
    dec = *reinterpret_cast<const f32x4*>(p.decay + c0 + cl);
  }
  __syncthreads();   // meta is there
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) {
    const RowMeta& r = L.meta[mi * 16 + r16];
    S0[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (wvalid && r.seq >= 0 && r.first && r.ctx > 0) S0[mi] = *reinterpret_cast<const f32x4*>(p.state + (int64_t)r.slot * p.width + c0 + cl);
  }
  constexpr int YU = (BM * (CT / 8) + 255) / 256;   // this thread's units of the output: y
  V8<T> yv[YU];
#pragma unroll
  for (int i = 0; i < YU; ++i) {
    const int m = (tid + i * 256) / (CT / 8), k = ((tid + i * 256) % (CT / 8)) * 8;
    yv[i] = load8(static_cast<const T*>(p.yx) + (int64_t)(t0 + min(m, rows - 1)) * p.ldx + c0 + min(k, nch - 8));
  }
  for (int k0 = 0; k0 < bw; k0 += KCH) {
    const int kn = min(KCH, bw - k0);
    // the chunk's first gate tiles are in flight while u is computed: all of them for few rows, four k-steps for many (more would cost the second workgroup; in 32 bits four spill), the
    // others behind them.  Blocks of 256, width 2048, 2773 rows 47.9 -> 43.6 us, 1024 rows 21.6 -> 21.1; 1024, 2115 rows 22.6 -> 21.8
    constexpr int AHEAD = BM == 16 ? KCH / 32 : sizeof(T) == 2 ? 4 : 2;
    V8<T> fr[AHEAD], fi[AHEAD];
    auto load_gates = [&](int i, int k) {
      const int64_t at = (int64_t)((k0 >> 5) + min(k, (kn >> 5) - 1)) * 512;
      fr[i] = load8(wr + at), fi[i] = load8(wi + at);
    };
    if (wvalid) {
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) load_gates(k, k);
    }
    if (k0 > 0) __syncthreads();   // the previous chunk has been read
    auto conv_row = [&](int m, int k) {
      const RowMeta& r = L.meta[m];
      if (r.seq >= 0 && k < kn) *reinterpret_cast<V8<T>*>(L.u + m * LDU + k) = from_f32<T>(conv8<T, TAPS>(p, r, t0 + m, blk * bw + k0 + k));
      else if (k < kn) *reinterpret_cast<V8<T>*>(L.u + m * LDU + k) = zero8<T>();
    };
    if constexpr (BM == 64 && TAPS > 0) {
      // eight channels of eight consecutive rows: inside one portion, past its first taps, the rows share their inputs
      const int k = (tid % (KCH / 8)) * 8, m0 = (tid / (KCH / 8)) * 8;
      const RowMeta &ra = L.meta[m0], &rb = L.meta[m0 + 7];
      if (k < kn && ra.seq >= 0 && ra.seq == rb.seq && t0 + m0 - (TAPS - 1) >= ra.qs) {
        const int c = blk * bw + k0 + k;
        const T* in = static_cast<const T*>(p.yx) + (int64_t)(t0 + m0 - (TAPS - 1)) * p.ldx + p.width + c;
        V8<T> v[TAPS + 7];
        f32x8 w[TAPS];
#pragma unroll
        for (int j = 0; j < TAPS + 7; ++j) v[j] = load8(in + (int64_t)j * p.ldx);
#pragma unroll
        for (int j = 0; j < TAPS; ++j) w[j] = load8(p.conv_w + (int64_t)j * p.width + c);
        const f32x8 b = load8(p.conv_b + c);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          f32x8 acc = b;
#pragma unroll
          for (int j = 0; j < TAPS; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] = fmaf(w[j][e], (float)v[m + j][e], acc[e]);
          *reinterpret_cast<V8<T>*>(L.u + (m0 + m) * LDU + k) = from_f32<T>(acc);
        }
      } else {
#pragma unroll 1
        for (int m = 0; m < 8; ++m) conv_row(m0 + m, k);
      }
    } else {
#pragma unroll 2
      for (int u = tid; u < BM * (KCH / 8); u += 256) conv_row(u / (KCH / 8), (u % (KCH / 8)) * 8);
    }
    __syncthreads();
    if (wvalid) {
      auto product = [&](int k, const V8<T>& a, const V8<T>& b) {
#pragma unroll
        for (int mi = 0; mi < MT; ++mi) {
          const V8<T> fu = load8(L.u + (mi * 16 + r16) * LDU + k * 32 + 8 * kc);
          mma(ar[mi], a, fu);
          mma(ai[mi], b, fu);
        }
      };
#pragma unroll
      for (int k = 0; k < KCH / 32; ++k) {
        if (k < kn >> 5) product(k, fr[k % AHEAD], fi[k % AHEAD]);
        if (k + AHEAD < KCH / 32) load_gates(k % AHEAD, k + AHEAD);
      }
    }
  }
  // the workgroup's own channels of u: into b, from LDS or (a block of several chunks) computed again
  const bool held = bw <= KCH;
  if (held) __syncthreads();
  for (int u = tid; u < BM * (CT / 8); u += 256) {
    const int m = u / (CT / 8), k = (u % (CT / 8)) * 8;
    const RowMeta& r = L.meta[m];
    f32x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
    if (held && k < nch) v = to_f32<T>(load8(L.u + m * LDU + cin + k));
    else if (r.seq >= 0 && k < nch) v = to_f32<T>(from_f32<T>(conv8<T, TAPS>(p, r, t0 + m, c0 + k)));   // rounded as the gates saw it
    *reinterpret_cast<f32x8*>(L.b + m * LDA + k) = v;
  }
  __syncthreads();
  if (wvalid) {
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
      const int m = mi * 16 + r16;
      const RowMeta& r = L.meta[m];
      const f32x4 u = *reinterpret_cast<const f32x4*>(L.b + m * LDA + cl);
      f32x4 a, b;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float la = dec[e] * sigmoid(ar[mi][e] + br[e]);
        a[e] = exp_hw(la);
        b[e] = __builtin_amdgcn_sqrtf(one_minus_exp(-2.f * la, a[e] * a[e])) * sigmoid(ai[mi][e] + bi[e]) * u[e];
        if (r.seq < 0) a[e] = 1.f, b[e] = 0.f;
        if (r.first) {
          b[e] = fmaf(a[e], S0[mi][e], b[e]);
          a[e] = 0.f;
        }
      }
      *reinterpret_cast<f32x4*>(L.a + m * LDA + cl) = a;
      *reinterpret_cast<f32x4*>(L.b + m * LDA + cl) = b;
    }
  }
  __syncthreads();
  const bool lead0 = L.meta[0].seq >= 0 && !L.meta[0].first;   // the tile opens inside a portion
  if (!p.single) {   // the walk, in place (b becomes S, a becomes P): a wave takes a quarter of the rows, a lane a channel
    constexpr int RW = BM / 4;
    float* pa = L.a + wave * RW * LDA + lane;
    float* pb = L.b + wave * RW * LDA + lane;
    if (lane < nch) {
      float S = 0.f, P = wave == 0 ? (lead0 ? 1.f : 0.f) : 1.f;
#pragma unroll 8
      for (int m = 0; m < RW; ++m) {
        const float a = pa[m * LDA], b = pb[m * LDA];
        S = fmaf(a, S, b);
        P *= a;
        pb[m * LDA] = S;
        pa[m * LDA] = P;
      }
      L.end[0][wave][lane] = S;
      L.end[1][wave][lane] = P;
    }
    __syncthreads();
    if (lane < nch && wave > 0) {   // what the quarters before this one hand over
      float S = L.end[0][0][lane], P = L.end[1][0][lane];
      for (int w = 1; w < wave; ++w) {
        S = fmaf(L.end[1][w][lane], S, L.end[0][w][lane]);
        P *= L.end[1][w][lane];
      }
#pragma unroll 8
      for (int m = 0; m < RW; ++m) {
        pb[m * LDA] = fmaf(pa[m * LDA], S, pb[m * LDA]);
        pa[m * LDA] *= P;
      }
    }
  }
  __syncthreads();
  const int lead_end = lead0 ? min(rows, L.meta[0].qs + L.meta[0].len - t0) : 0;   // rows of the leading segment
#pragma unroll
  for (int i = 0; i < YU; ++i) {
    const int u = tid + i * 256, m = u / (CT / 8), k = (u % (CT / 8)) * 8;
    if (m >= rows || k >= nch) continue;
    const RowMeta& r = L.meta[m];
    const f32x8 S = *reinterpret_cast<const f32x8*>(L.b + m * LDA + k);
    const int t = t0 + m, c = c0 + k;
    if (r.seq < 0) {
      *reinterpret_cast<V8<T>*>(static_cast<T*>(p.out) + (int64_t)t * p.ldo + c) = zero8<T>();
      continue;
    }
    const bool lead = m < lead_end;
    if (lead || (m == BM - 1 && !r.last)) {   // unfinished, or what the next tile's carry starts from
      *reinterpret_cast<f32x8*>(p.scratch + (int64_t)t * p.width + c) = S;
      *reinterpret_cast<f32x8*>(p.scratch + ((int64_t)s.T + t) * p.width + c) = *reinterpret_cast<const f32x8*>(L.a + m * LDA + k);
    }
    if (lead) continue;
    store_out8<T>(p, t, c, S, to_f32<T>(yv[i]));
    if (r.last) *reinterpret_cast<f32x8*>(p.state + (int64_t)r.slot * p.width + c) = S;
  }
  // the convolution tail of entries that end in this tile, into its other half
  const int nt = p.taps - 1;
  for (int u = tid; u < rows * nt * (CT / 8); u += 256) {
    const int k = (u % (CT / 8)) * 8, e = u / (CT / 8) % nt, m = u / (CT / 8) / nt, c = c0 + k;
    const RowMeta& r = L.meta[m];
    if (k >= nch || r.seq < 0 || !r.last) continue;
    const T* from = static_cast<const T*>(p.tail) + ((int64_t)r.slot * 2 + r.flip) * nt * p.width;
    T* to = static_cast<T*>(p.tail) + ((int64_t)r.slot * 2 + (r.flip ^ 1)) * nt * p.width;
    const int pos = r.ctx + r.len - nt + e;   // the position this entry stands for
    V8<T> v = zero8<T>();
    if (pos >= r.ctx) v = load8(static_cast<const T*>(p.yx) + (int64_t)(r.qs + pos - r.ctx) * p.ldx + p.width + c);
    else if (pos >= 0) v = load8(from + (int64_t)(pos - (r.ctx - nt)) * p.width + c);
    *reinterpret_cast<V8<T>*>(to + (int64_t)e * p.width + c) = v;
  }
}

// carries from tile to tile of the entries that span tiles: one thread per (entry, channel)
__global__ __launch_bounds__(64) void rglru_carry_kernel(const vmi_hy_rglru_args p, const vmi_hy_step s) {
  constexpr int BM = 64;
  const int c = blockIdx.x * 64 + threadIdx.x, q = blockIdx.y;
  if (c >= p.width || s.q_len[q] <= 0) return;
  const int qs = s.q_start[q], qe = qs + s.q_len[q];
  const int first = qs / BM, last = (qe - 1) / BM;
  if (first == last) return;
  const float* S = p.scratch + c;
  const float* P = p.scratch + (int64_t)s.T * p.width + c;
  float carry = S[(int64_t)(first * BM + BM - 1) * p.width];
  constexpr int U = 8;
  for (int k = first + 1; k <= last; k += U) {
    float sv[U], pv[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int64_t row = min((k + i) * BM + BM, qe) - 1;
      sv[i] = k + i <= last ? S[row * p.width] : 0.f;
      pv[i] = k + i <= last ? P[row * p.width] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      if (k + i <= last) {
        p.carry[(int64_t)(k + i) * p.width + c] = carry;
        carry = fmaf(pv[i], carry, sv[i]);
      }
    }
  }
  p.state[(int64_t)s.state_slot[q] * p.width + c] = carry;
}

// the rows of leading segments: S + P * carry
template <typename T>
__global__ __launch_bounds__(256) void rglru_finish_kernel(const vmi_hy_rglru_args p, const vmi_hy_step s) {
  constexpr int BM = 64;
  const int t = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * 8;
  const int q = s.tok_seq[t];
  if (c >= p.width || q < 0) return;
  const int tile = t / BM;
  if (s.q_start[q] >= tile * BM) return;
  const f32x8 S = load8(p.scratch + (int64_t)t * p.width + c), P = load8(p.scratch + ((int64_t)s.T + t) * p.width + c);
  const f32x8 k = load8(p.carry + (int64_t)tile * p.width + c);
  f32x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = fmaf(P[e], k[e], S[e]);
  store_out8<T>(p, t, c, o, to_f32<T>(load8(static_cast<const T*>(p.yx) + (int64_t)t * p.ldx + c)));
}

// A step of single tokens, bfloat16.  A workgroup takes 16 tokens x NO tiles of 16 channels of one gate block; its eight waves share the block's channels, the k of
// the gate products: a lane convolves eight channels of one token, which is the products' operand as it stands, so nothing goes through LDS but the partial products
// and the workgroup's own channels.  Tokens are their entries, so what the tables say of a token is asked for at once.  Bound by three trips through memory
// (tables, states and tails, results) and the launch; rglru_tile_kernel's workgroups, 64 channels each, left most of the chip idle.  Blocks of
// 256, width 1024, 1 / 12 / 64 tokens 5.7 / 6.7 / 6.9 -> 4.3 / 4.6 / 5.3 us, width 4096, 1 / 12 / 64 5.7 / 7.7 / 8.4 -> 4.4 / 5.3 / 6.8.
template <int NO, int TAPS>   // TAPS = 0: any number of taps
__global__ __launch_bounds__(512, 2) void rglru_step_kernel(const vmi_hy_rglru_args p, const vmi_hy_step s) {
  constexpr int RW = 8, LDU = NO * 16 + 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  f32x4* part = reinterpret_cast<f32x4*>(smem);                     // [RW][NO][2][64]
  b16* own = reinterpret_cast<b16*>(part + RW * NO * 2 * 64);       // [16][LDU]: this workgroup's channels behind the convolution
  need(p.yx), need(p.out), need(p.conv_w), need(p.conv_b), need(p.gates), need(p.gate_b), need(p.decay), need(p.state), need(p.tail), need(p.ldx), need(p.ldo), need(p.width),
      need(p.blocks), need(s.tok_seq), need(s.ctx), need(s.state_slot), need(s.flip), need(s.T), need(s.B);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kc = lane >> 4, r16 = lane & 15;
  const int taps = TAPS ? TAPS : p.taps, nt = taps - 1;
  const int bw = p.width / p.blocks, nks = bw >> 5, tiles = bw >> 4, ng = (tiles + NO - 1) / NO;
  const int blk = blockIdx.x / ng, o0 = blockIdx.x % ng * NO, t0 = blockIdx.y * 16, rows = min(16, s.T - t0);
  struct Row {
    int seq, ctx, slot, flip;
  };
  auto row_of = [&](int m) {
    const int t = t0 + min(m, rows - 1), e = min(t, s.B - 1);
    Row r{s.tok_seq[t], s.ctx[e], s.state_slot[e], s.flip[e]};
    if (r.seq >= 0 && r.seq != e) r.ctx = s.ctx[r.seq], r.slot = s.state_slot[r.seq], r.flip = s.flip[r.seq];   // (tokens in another order than entries)
    if (r.seq < 0) r.ctx = r.slot = r.flip = 0;   // (a padding row's entry may hold anything: it reads the first state and stores none)
    return r;
  };
  const b16* yx = static_cast<const b16*>(p.yx);
  const b16* tail = static_cast<const b16*>(p.tail);
  const int t = t0 + min(r16, rows - 1);

  // what needs no table: this lane's inputs and weights of its wave's first k-step, the gates' tiles, what the results need
  auto channel = [&](int ks) { return blk * bw + 32 * min(ks, nks - 1) + 8 * kc; };
  V8<b16> x = load8(yx + (int64_t)t * p.ldx + p.width + channel(wave));
  const b16* gp = static_cast<const b16*>(p.gates) + (int64_t)blk * bw * bw + lane * 8;
  const int64_t gsz = (int64_t)p.blocks * bw * bw;
  b16x8 gr[NO], gi[NO];
  auto load_gates = [&](int ks) {
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      const int64_t at = ((int64_t)min(o0 + o, tiles - 1) * nks + min(ks, nks - 1)) * 512;
      gr[o] = load8(gp + at), gi[o] = load8(gp + gsz + at);
    }
  };
  const Row mine = row_of(r16);
  f32x8 cw[TAPS ? TAPS : 1], cb = load8(p.conv_b + channel(wave));
  if constexpr (TAPS > 0) {
#pragma unroll
    for (int j = 0; j < TAPS; ++j) cw[j] = load8(p.conv_w + (int64_t)j * p.width + channel(wave));
  }
  load_gates(wave);
  const bool ends = wave < NO && o0 + wave < tiles;   // whether this wave finishes a tile, and which of its channels this lane does
  const int c = blk * bw + min(o0 + wave, tiles - 1) * 16 + 4 * kc;
  f32x4 br, bi, dec, S0;
  b16x4 y;
  if (ends) {
    br = *reinterpret_cast<const f32x4*>(p.gate_b + c);
    bi = *reinterpret_cast<const f32x4*>(p.gate_b + p.width + c);
    dec = *reinterpret_cast<const f32x4*>(p.decay + c);
    y = *reinterpret_cast<const b16x4*>(yx + (int64_t)t * p.ldx + c);
  }
  const bool live = mine.seq >= 0;
  const b16* old = tail + ((int64_t)mine.slot * 2 + mine.flip) * nt * p.width;
  if (ends) S0 = *reinterpret_cast<const f32x4*>(p.state + (int64_t)mine.slot * p.width + c);

  f32x4 ar[NO], ai[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) ar[o] = ai[o] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int ks = wave; ks < nks; ks += RW) {
    const int ch = channel(ks);
    f32x8 acc;
    if constexpr (TAPS > 0) {
      if (ks > wave) {
        x = load8(yx + (int64_t)t * p.ldx + p.width + ch);
        cb = load8(p.conv_b + ch);
#pragma unroll
        for (int j = 0; j < TAPS; ++j) cw[j] = load8(p.conv_w + (int64_t)j * p.width + ch);
        load_gates(ks);
      }
      b16x8 v[TAPS];
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) v[j] = load8(old + (int64_t)j * p.width + ch);
      v[TAPS - 1] = x;
      acc = cb;
#pragma unroll
      for (int j = 0; j < TAPS; ++j) {
        const bool on = mine.ctx >= TAPS - 1 - j;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = fmaf(cw[j][e], on ? (float)v[j][e] : 0.f, acc[e]);
      }
    } else {
      if (ks > wave) load_gates(ks);
      acc = load8(p.conv_b + ch);
      for (int j = 0; j < taps; ++j) {
        const b16x8 v = load8(j < nt ? old + (int64_t)j * p.width + ch : yx + (int64_t)t * p.ldx + p.width + ch);
        const f32x8 w = load8(p.conv_w + (int64_t)j * p.width + ch);
        const bool on = mine.ctx >= nt - j;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = fmaf(w[e], on ? (float)v[e] : 0.f, acc[e]);
      }
    }
    const b16x8 u = live ? from_f32<b16>(acc) : zero8<b16>();
    const int k = 32 * ks + 8 * kc - o0 * 16;
    if (k >= 0 && k < NO * 16) *reinterpret_cast<b16x8*>(own + r16 * LDU + k) = u;
#pragma unroll
    for (int o = 0; o < NO; ++o) mma(ar[o], gr[o], u), mma(ai[o], gi[o], u);
  }
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    part[((wave * NO + o) * 2) * 64 + lane] = ar[o];
    part[((wave * NO + o) * 2 + 1) * 64 + lane] = ai[o];
  }
  // the convolution's tail, into its other half
  for (int u = tid; u < rows * nt * 2 * NO; u += 512) {
    const int k = u % (2 * NO), e = u / (2 * NO) % nt, m = u / (2 * NO) / nt, ch = blk * bw + o0 * 16 + k * 8;
    const Row r = row_of(m);
    if (r.seq < 0 || o0 * 16 + k * 8 >= bw) continue;
    const int64_t at = ((int64_t)r.slot * 2 + r.flip) * nt * p.width + ch, to = ((int64_t)r.slot * 2 + (r.flip ^ 1)) * nt * p.width + ch;
    const int pos = r.ctx + 1 - nt + e;   // the position this entry stands for
    V8<b16> v = zero8<b16>();
    if (e == nt - 1) v = load8(yx + (int64_t)(t0 + m) * p.ldx + p.width + ch);
    else if (pos >= 0) v = load8(tail + at + (int64_t)(e + 1) * p.width);
    *reinterpret_cast<V8<b16>*>(static_cast<b16*>(p.tail) + to + (int64_t)e * p.width) = v;
  }
  __syncthreads();
  if (!ends || r16 >= rows) return;
  f32x4 sr = part[(wave * 2) * 64 + lane], si = part[(wave * 2 + 1) * 64 + lane];
#pragma unroll
  for (int w = 1; w < RW; ++w) sr += part[((w * NO + wave) * 2) * 64 + lane], si += part[((w * NO + wave) * 2 + 1) * 64 + lane];
  const b16x4 u = *reinterpret_cast<const b16x4*>(own + r16 * LDU + wave * 16 + 4 * kc);
  f32x4 S;
  b16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float la = dec[e] * sigmoid(sr[e] + br[e]), a = exp_hw(la);
    const float b = __builtin_amdgcn_sqrtf(one_minus_exp(-2.f * la, a * a)) * sigmoid(si[e] + bi[e]) * (float)u[e];
    S[e] = fmaf(a, mine.ctx > 0 ? S0[e] : 0.f, b);
    o[e] = live ? (b16)(S[e] * gelu_tanh((float)y[e])) : (b16)0.f;
  }
  *reinterpret_cast<b16x4*>(static_cast<b16*>(p.out) + (int64_t)(t0 + r16) * p.ldo + c) = o;
  if (live) *reinterpret_cast<f32x4*>(p.state + (int64_t)mine.slot * p.width + c) = S;
}

template <int NO>
static int launch_step(const vmi_hy_rglru_args& p, const vmi_hy_step& s, hipStream_t st) {
  auto* fn = p.taps == 4 ? rglru_step_kernel<NO, 4> : rglru_step_kernel<NO, 0>;
  const size_t lds = (size_t)8 * NO * 2 * 1024 + (size_t)16 * (NO * 16 + 8) * 2;
  if (int rc = allow_lds(fn, lds, "vmi_hy_rglru")) return rc;
  const int tiles = p.width / p.blocks / 16;
  hipLaunchKernelGGL(fn, dim3(p.blocks * ((tiles + NO - 1) / NO), (s.T + 15) / 16), dim3(512), lds, st, p, s);
  return launched("vmi_hy_rglru");
}

template <typename T, int BM, int TAPS>
static int launch_tile(const vmi_hy_rglru_args& p, const vmi_hy_step& s, hipStream_t st) {
  auto* fn = rglru_tile_kernel<T, BM, TAPS>;
  if (int rc = allow_lds(fn, sizeof(Lds<T, BM>), "vmi_hy_rglru")) return rc;
  const int bw = p.width / p.blocks;
  hipLaunchKernelGGL(fn, dim3(p.blocks * ((bw + CT - 1) / CT), (s.T + BM - 1) / BM), dim3(256), sizeof(Lds<T, BM>), st, p, s);
  return launched("vmi_hy_rglru");
}

template <typename T>
static int run_rglru(const vmi_hy_rglru_args& p, const vmi_hy_step& s, hipStream_t st) {
  if constexpr (sizeof(T) == 2) {
    // as few tiles a workgroup as leave one of them a compute unit, each convolves all of its block's channels; past four, rglru_tile_kernel's 64 channels beside rows in
    // LDS are as good (width 2048, 256 tokens, 2048 tiles 10.2 us, here 11.2; width 4096, 64 tokens, 1024 tiles 8.4 and 6.8)
    const int64_t n = (int64_t)(p.width / 16) * ((s.T + 15) / 16);
    if (p.single && n <= 1024) return n <= 256 ? launch_step<1>(p, s, st) : n <= 512 ? launch_step<2>(p, s, st) : launch_step<4>(p, s, st);
  }
  if (p.single) {
    return p.taps == 4 ? launch_tile<T, 16, 4>(p, s, st) : launch_tile<T, 16, 0>(p, s, st);
  }
  if (int rc = p.taps == 4 ? launch_tile<T, 64, 4>(p, s, st) : launch_tile<T, 64, 0>(p, s, st)) return rc;
  if (!p.spans) return VMI_HY_OK;
  hipLaunchKernelGGL(rglru_carry_kernel, dim3((p.width + 63) / 64, s.B), dim3(64), 0, st, p, s);
  hipLaunchKernelGGL(rglru_finish_kernel<T>, dim3((p.width / 8 + 255) / 256, s.T), dim3(256), 0, st, p, s);
  return launched("vmi_hy_rglru");
}

}  // namespace vmi_hybrid

using namespace vmi_hybrid;

extern "C" int vmi_hy_rglru(const vmi_hy_rglru_args* a, const vmi_hy_step* s, void* stream) {
  static const char* who = "vmi_hy_rglru";
  if (!a || !s || !a->yx || !a->out || !a->conv_w || !a->conv_b || !a->gates || !a->gate_b || !a->decay || !a->state ||
      (a->taps > 1 && !a->tail) || !s->tok_seq || !s->q_start || !s->q_len || !s->ctx || !s->state_slot || !s->flip || s->T <= 0 ||
      s->B <= 0 || a->width <= 0 || a->blocks <= 0 || a->taps < 1 || (a->spans && (!a->scratch || !a->carry)))
    return fail(VMI_HY_E_ARG, who, "null pointer or non-positive size");
  if (a->width % a->blocks || ((a->width / a->blocks) & 31) || (a->ldx & 7) || (a->ldo & 7) || a->taps > MAX_TAPS || s->T > 65535 * 16 ||
      (a->spans && s->T > 65535))
    return fail(VMI_HY_E_SHAPE, who, "needs blocks of a multiple of 32 channels, rows of a multiple of 8 elements, at most 16 taps");
  if (!a->single && !a->spans && !a->scratch) return fail(VMI_HY_E_ARG, who, "portions need scratch");
  DeviceScope dev(a->device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  return a->dtype == VMI_HY_BF16 ? run_rglru<b16>(*a, *s, st) : run_rglru<float>(*a, *s, st);
}
