// The recurrent block between its projections (include/vmi_hybrid.h): causal convolution -> block-diagonal gates -> gated linear
// recurrence -> product with gelu(y).
//
// The packed tokens are cut into row tiles of BM consecutive rows, whatever entries they belong to.  A workgroup takes one row
// tile x up to CT channels of one gate block: the convolution of the block's channels goes to LDS (element type), both gate
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

constexpr int KCH = 256;    // channels of u in LDS at a time
constexpr int MAX_TAPS = 16;

struct RowMeta {
  int seq, qs, len, ctx, slot, flip, first, last;
};

template <typename T, int BM, int CT>
struct Lds {
  static constexpr int LDU = KCH + 16 / (int)sizeof(T), LDA = CT + 4;
  union {   // u until the gates' products are done, then the states
    T u[BM * LDU];
    float S[BM * LDA];
  };
  RowMeta meta[BM];
};

// Lane 15's value to the 16 lanes of its row.
__device__ __forceinline__ float lane15(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x15f, 0xf, 0xf, true));
}
// Four recurrences S = A S + B over the 16 lanes of a row, in place: the lane D below's pair (0 and unchanged where there is none) in front of a lane's own, D = 1, 2, 4, 8.  As
// builtins a step was six instructions a value, of them four moves; here it is two, and each is eight behind the one whose result it takes from another lane (two are asked for).
__device__ __forceinline__ void walk16(f32x4& A, f32x4& B) {
  float a0 = A[0], a1 = A[1], a2 = A[2], a3 = A[3], b0 = B[0], b1 = B[1], b2 = B[2], b3 = B[3];
#define VMI_STEP(D)                                                                 \
  "v_fmac_f32_dpp %4, %4, %0 row_shr:" #D " row_mask:0xf bank_mask:0xf bound_ctrl:0\n" \
  "v_fmac_f32_dpp %5, %5, %1 row_shr:" #D " row_mask:0xf bank_mask:0xf bound_ctrl:0\n" \
  "v_fmac_f32_dpp %6, %6, %2 row_shr:" #D " row_mask:0xf bank_mask:0xf bound_ctrl:0\n" \
  "v_fmac_f32_dpp %7, %7, %3 row_shr:" #D " row_mask:0xf bank_mask:0xf bound_ctrl:0\n" \
  "v_mul_f32_dpp %0, %0, %0 row_shr:" #D " row_mask:0xf bank_mask:0xf\n"               \
  "v_mul_f32_dpp %1, %1, %1 row_shr:" #D " row_mask:0xf bank_mask:0xf\n"               \
  "v_mul_f32_dpp %2, %2, %2 row_shr:" #D " row_mask:0xf bank_mask:0xf\n"               \
  "v_mul_f32_dpp %3, %3, %3 row_shr:" #D " row_mask:0xf bank_mask:0xf\n"
  asm("s_nop 1\n" VMI_STEP(1) VMI_STEP(2) VMI_STEP(4) VMI_STEP(8)
      "s_nop 1"
      : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3));
#undef VMI_STEP
  A = f32x4{a0, a1, a2, a3}, B = f32x4{b0, b1, b2, b3};
}

// The same where a value is no finite number: a zero of A stops what is in front of it, whatever that is.  first: whether a lane's row opens a portion (A is 0 there); afterwards, whether one of its
// lanes up to this one does.  Slower by an instruction or three a value, for the rare wave whose portions would else meet.
template <int D>
__device__ __forceinline__ void step16(f32x4& A, f32x4& B, int& first) {
  auto below = [](float old, float v) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, v), 0x110 + D, 0xf, 0xf, false)); };
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = below(1.f, A[e]), b = below(0.f, B[e]);
    B[e] = first ? B[e] : fmaf(A[e], b, B[e]);
    A[e] = first ? A[e] : A[e] * a;
  }
  first |= __builtin_amdgcn_update_dpp(0, first, 0x110 + D, 0xf, 0xf, false);
}

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
#pragma unroll 1
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

// CT channels of one gate block to a workgroup, 16 to a wave.  A lane's gate results are four channels of one row of each 16, so the walk over a tile stays in registers: four
// doubling steps across the 16 lanes of a row group, then group after group through lane 15.
// Bound by the instructions of a wave, some 2500 of them issued one by one (two waves a SIMD, whose registers no more fit: at 128 they spill), and by five trips to memory in front
// of them.  So 128 channels (each workgroup of a block convolves all of its channels, 64 do so twice as often), inputs and weights asked for before the tables are there, a portion's
// first rows from the same registers as its others (they went one by one), and no walk through LDS (16 rows a wave, twice, four barriers).  us, blocks of 256: width 1024, 6 x 20
// tokens 18.7 -> 14.1, 48 x 80 22.2 -> 15.5, 4 x up to 1000 25.1 -> 24.5; 2048, 4 x up to 1024 43.0 -> 38.5, 40 x 100 39.6 -> 28.9; 4096, 4 x 300 32.1 -> 26.3.
template <typename T, int BM, int TAPS, int CT>
__global__ __launch_bounds__(4 * CT, 2) void rglru_tile_kernel(const vmi_hy_rglru_args p, const vmi_hy_step s) {
  constexpr int MT = BM / 16, TH = 4 * CT;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  auto& L = *reinterpret_cast<Lds<T, BM, CT>*>(smem);
  constexpr int LDU = Lds<T, BM, CT>::LDU, LDA = Lds<T, BM, CT>::LDA;
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
  f32x4 br, bi, dec;
  if (wvalid) {
    br = *reinterpret_cast<const f32x4*>(p.gate_b + c0 + cl);
    bi = *reinterpret_cast<const f32x4*>(p.gate_b + p.width + c0 + cl);
    dec = *reinterpret_cast<const f32x4*>(p.decay + c0 + cl);
  }
  // eight channels of this many consecutive rows to a thread: past the taps of their portions' starts they share their inputs, which need no table to be asked for
  constexpr bool TOGETHER = BM == 64 && TAPS > 0;
  constexpr int RPT = TOGETHER ? BM * (KCH / 8) / TH : 1;
  const int kr = (tid % (KCH / 8)) * 8, m0 = tid / (KCH / 8) * RPT;
  V8<T> v[TOGETHER ? TAPS - 1 + RPT : 1];
  f32x8 w[TOGETHER ? TAPS : 1], wb;
  auto ask = [&](int k0) {
    if constexpr (TOGETHER) {
      const int c = blk * bw + k0 + min(kr, min(KCH, bw - k0) - 8);
#pragma unroll
      for (int j = 0; j < TAPS; ++j) w[j] = load8(p.conv_w + (int64_t)j * p.width + c);
      wb = load8(p.conv_b + c);
      const T* in = static_cast<const T*>(p.yx) + p.width + blk * bw + k0 + min(kr, min(KCH, bw - k0) - 8);
#pragma unroll
      for (int j = 0; j < TAPS - 1 + RPT; ++j) v[j] = load8(in + (int64_t)min(max(t0 + m0 - (TAPS - 1) + j, 0), s.T - 1) * p.ldx);
    }
  };
  constexpr bool SOON = sizeof(T) == 2;   // (in 32 bits they spill)
  if constexpr (SOON) ask(0);
  __syncthreads();   // meta is there
  constexpr int YU = (BM * (CT / 8) + TH - 1) / TH;   // this thread's units of the output: y
  V8<T> yv[YU];
#pragma unroll
  for (int i = 0; i < YU; ++i) {
    const int m = (tid + i * TH) / (CT / 8), k = ((tid + i * TH) % (CT / 8)) * 8;
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
    if (!SOON || k0 > 0) ask(k0);
    if (k0 > 0) __syncthreads();   // the previous chunk has been read
    auto conv_row = [&](int m, int k) {   // (beside rows that are taken together: the loop over taps, whose registers they need)
      const RowMeta& r = L.meta[m];
      if (r.seq >= 0 && k < kn) *reinterpret_cast<V8<T>*>(L.u + m * LDU + k) = from_f32<T>(conv8<T, TOGETHER ? 0 : TAPS>(p, r, t0 + m, blk * bw + k0 + k));
      else if (k < kn) *reinterpret_cast<V8<T>*>(L.u + m * LDU + k) = zero8<T>();
    };
    if constexpr (TOGETHER) {
      const RowMeta &ra = L.meta[m0], &rb = L.meta[m0 + RPT - 1];
      const bool inside = ra.seq >= 0 && ra.seq == rb.seq && t0 + m0 - (TAPS - 1) >= ra.qs;
      bool tails = false;   // whether a row's taps reach into what its sequence had before
      if (!inside) {
#pragma unroll
        for (int m = 0; m < RPT; ++m) {
          const RowMeta& r = L.meta[m0 + m];
          tails |= r.seq >= 0 && r.ctx > 0 && t0 + m0 + m - (TAPS - 1) < r.qs;
        }
      }
      if (k0 + kr < k0 + kn && !tails) {
#pragma unroll
        for (int m = 0; m < RPT; ++m) {
          f32x8 acc = wb;
          const int back = inside ? TAPS - 1 : L.meta[m0 + m].seq < 0 ? -1 : min(t0 + m0 + m - L.meta[m0 + m].qs, TAPS - 1);   // rows of this portion before this one
#pragma unroll
          for (int j = 0; j < TAPS; ++j)
            if (TAPS - 1 - j <= back) {
#pragma unroll
              for (int e = 0; e < 8; ++e) acc[e] = fmaf(w[j][e], (float)v[m + j][e], acc[e]);
            }
          *reinterpret_cast<V8<T>*>(L.u + (m0 + m) * LDU + kr) = back < 0 ? zero8<T>() : from_f32<T>(acc);
        }
      } else if (kr < kn) {
#pragma unroll 1
        for (int m = 0; m < RPT; ++m) conv_row(m0 + m, kr);
      }
    } else {
#pragma unroll 2
      for (int u = tid; u < BM * (KCH / 8); u += TH) conv_row(u / (KCH / 8), (u % (KCH / 8)) * 8);
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
  // the workgroup's own channels of u are in LDS, or (a block of several chunks) computed again
  const bool held = bw <= KCH;
  if (!held) {
    __syncthreads();
    for (int u = tid; u < BM * (CT / 8); u += TH) {
      const int m = u / (CT / 8), k = (u % (CT / 8)) * 8;
      const RowMeta& r = L.meta[m];
      V8<T> x = zero8<T>();
      if (r.seq >= 0 && k < nch) x = from_f32<T>(conv8<T, TOGETHER ? 0 : TAPS>(p, r, t0 + m, c0 + k));   // rounded as the gates saw it
      *reinterpret_cast<V8<T>*>(L.u + m * LDU + k) = x;
    }
    __syncthreads();
  }
  const bool lead0 = L.meta[0].seq >= 0 && !L.meta[0].first;   // the tile opens inside a portion
  const int lead_end = lead0 ? min(rows, L.meta[0].qs + L.meta[0].len - t0) : 0;   // rows of the leading segment
  // a row that is unfinished, or what the next tile's carry starts from: its state and product go to scratch
  auto kept = [&](int m, const RowMeta& r) { return m < rows && r.seq >= 0 && (m < lead_end || (m == BM - 1 && !r.last)); };
  f32x4 Sc{0.f, 0.f, 0.f, 0.f}, Pc;
  Pc[0] = Pc[1] = Pc[2] = Pc[3] = lead0 ? 1.f : 0.f;
  if (wvalid) {
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
      const int m = mi * 16 + r16;
      const RowMeta& r = L.meta[m];
      const T* u = L.u + m * LDU + (held ? cin : 0) + cl;
      f32x4 &a = ar[mi], &b = ai[mi];
      const bool first = r.first, goes_on = first && r.ctx > 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {   // (a row that is no token's: u and with it b is 0, and what follows it opens a portion)
        const float la = dec[e] * sigmoid(a[e] + br[e]);
        a[e] = exp_hw(la);
        b[e] = __builtin_amdgcn_sqrtf(one_minus_exp(-2.f * la, a[e] * a[e])) * sigmoid(b[e] + bi[e]) * (float)u[e];
      }
      if (goes_on) b += a * *reinterpret_cast<const f32x4*>(p.state + (int64_t)r.slot * p.width + c0 + cl);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = first ? 0.f : a[e];
      if (!p.single) {
        float odd = 0.f;   // (0, or no number where one of these is none or infinite)
#pragma unroll
        for (int e = 0; e < 4; ++e) odd = fmaf(b[e], 0.f, fmaf(Sc[e], 0.f, odd));
        if (__builtin_amdgcn_ballot_w64(odd != odd) == 0) {   // (scalar)
          walk16(a, b);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            b[e] = fmaf(a[e], Sc[e], b[e]);
            a[e] *= Pc[e];
          }
        } else {
          int opened = first;
          step16<1>(a, b, opened), step16<2>(a, b, opened), step16<4>(a, b, opened), step16<8>(a, b, opened);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            b[e] = opened ? b[e] : fmaf(a[e], Sc[e], b[e]);
            a[e] = opened ? 0.f : a[e] * Pc[e];
          }
        }
        if (mi + 1 < MT) {
#pragma unroll
          for (int e = 0; e < 4; ++e) Sc[e] = lane15(b[e]), Pc[e] = lane15(a[e]);
        }
        if (kept(m, r)) *reinterpret_cast<f32x4*>(p.scratch + ((int64_t)s.T + t0 + m) * p.width + c0 + cl) = a;
      }
    }
  }
  __syncthreads();   // (u has been read)
  if (wvalid) {
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) *reinterpret_cast<f32x4*>(L.S + (mi * 16 + r16) * LDA + cl) = ai[mi];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < YU; ++i) {
    const int u = tid + i * TH, m = u / (CT / 8), k = (u % (CT / 8)) * 8;
    if (m >= rows || k >= nch) continue;
    const RowMeta& r = L.meta[m];
    const f32x8 S = *reinterpret_cast<const f32x8*>(L.S + m * LDA + k);
    const int t = t0 + m, c = c0 + k;
    if (r.seq < 0) {
      *reinterpret_cast<V8<T>*>(static_cast<T*>(p.out) + (int64_t)t * p.ldo + c) = zero8<T>();
      continue;
    }
    if (!p.single && kept(m, r)) *reinterpret_cast<f32x8*>(p.scratch + (int64_t)t * p.width + c) = S;
    if (m < lead_end) continue;
    store_out8<T>(p, t, c, S, to_f32<T>(yv[i]));
    if (r.last) *reinterpret_cast<f32x8*>(p.state + (int64_t)r.slot * p.width + c) = S;
  }
  // the convolution tail of entries that end in this tile, into its other half
  const int nt = p.taps - 1;
  for (int u = tid; u < rows * nt * (CT / 8); u += TH) {
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

// Both in one: a workgroup takes a row tile's leading segment and 256 channels, and runs the carry up to it itself.  Each tile so reads the ends of all tiles of its entry in front of
// it, which is less than a launch of its own takes up to MOST_TILES of them; beyond, that grows with their square.  rglru_carry_kernel + rglru_finish_kernel / here, us: width 2048, 1 x
// 130 rows 4.2 + 4.2 / 7.6, 4 x up to 1024 5.8 + 11.4 / 15.1, 40 x 100 4.3 + 6.5 / 10.0, 1 x 4096 15.2 + 16.5 / 25.3, x 8192 28.8 + 31.2 / 67.2; 1024, 1 x 4096 25.0 / 19.9, x 8192 43.5 / 37.8.
constexpr int MOST_TILES = 64;
template <typename T>
__global__ __launch_bounds__(256) void rglru_lead_kernel(const vmi_hy_rglru_args p, const vmi_hy_step s) {
  constexpr int BM = 64, U = 8;
  const int c = (blockIdx.x * 32 + threadIdx.x % 32) * 8, tile = blockIdx.y, t0 = tile * BM;
  const int q = s.tok_seq[t0];
  if (c >= p.width || q < 0) return;
  const int qs = s.q_start[q], qe = qs + s.q_len[q];
  if (qs >= t0) return;
  const float* S = p.scratch + c;
  const float* P = p.scratch + (int64_t)s.T * p.width + c;
  auto end_of = [&](int k) { return (int64_t)(k * BM + BM - 1) * p.width; };
  f32x8 carry = load8(S + end_of(qs / BM));
  for (int k = qs / BM + 1; k < tile; k += U) {
    f32x8 sv[U], pv[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {   // (past the last one: that one again)
      sv[i] = load8(S + end_of(min(k + i, tile - 1)));
      pv[i] = load8(P + end_of(min(k + i, tile - 1)));
    }
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (k + i < tile) {   // (scalar)
#pragma unroll
        for (int e = 0; e < 8; ++e) carry[e] = fmaf(pv[i][e], carry[e], sv[i][e]);
      }
  }
  const int end = min(t0 + BM, qe);
#pragma unroll 4
  for (int t = t0 + threadIdx.x / 32; t < end; t += 8) {
    const f32x8 a = load8(S + (int64_t)t * p.width), b = load8(P + (int64_t)t * p.width);
    const V8<T> y = load8(static_cast<const T*>(p.yx) + (int64_t)t * p.ldx + c);
    f32x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = fmaf(b[e], carry[e], a[e]);
    store_out8<T>(p, t, c, o, to_f32<T>(y));
    if (t == qe - 1) *reinterpret_cast<f32x8*>(p.state + (int64_t)s.state_slot[q] * p.width + c) = o;
  }
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

template <typename T, int BM, int TAPS, int CT>
static int launch_tile(const vmi_hy_rglru_args& p, const vmi_hy_step& s, hipStream_t st) {
  auto* fn = rglru_tile_kernel<T, BM, TAPS, CT>;
  if (int rc = allow_lds(fn, sizeof(Lds<T, BM, CT>), "vmi_hy_rglru")) return rc;
  const int bw = p.width / p.blocks;
  hipLaunchKernelGGL(fn, dim3(p.blocks * ((bw + CT - 1) / CT), (s.T + BM - 1) / BM), dim3(4 * CT), sizeof(Lds<T, BM, CT>), st, p, s);
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
    return p.taps == 4 ? launch_tile<T, 16, 4, 64>(p, s, st) : launch_tile<T, 16, 0, 64>(p, s, st);
  }
  constexpr int CT = sizeof(T) == 2 ? 128 : 64;   // (in 32 bits twice the channels spill twice the registers)
  const bool wide = CT > 64 && p.width / p.blocks > 64;
  if (int rc = p.taps == 4 ? (wide ? launch_tile<T, 64, 4, CT>(p, s, st) : launch_tile<T, 64, 4, 64>(p, s, st))
                           : (wide ? launch_tile<T, 64, 0, CT>(p, s, st) : launch_tile<T, 64, 0, 64>(p, s, st)))
    return rc;
  if (!p.spans) return VMI_HY_OK;
  if (const int tiles = (s.T + 63) / 64; tiles <= MOST_TILES) {
    hipLaunchKernelGGL(rglru_lead_kernel<T>, dim3((p.width / 8 + 31) / 32, tiles), dim3(256), 0, st, p, s);
    return launched("vmi_hy_rglru");
  }
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
