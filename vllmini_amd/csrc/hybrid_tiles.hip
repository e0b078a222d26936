// Products of many rows in bfloat16 with the gated unit behind them (mfma_tiles.hpp), include/vmi_hybrid.h: vmi_hy_linear_tiles.
#include "hybrid_common.hpp"
#include "hybrid_linear.hpp"
#include "mfma_tiles.hpp"

namespace vmi_hybrid {

// STORE_GLU: columns below n_split as they are, the others, interleaved (gate, up), through the gated unit: what a product and an elementwise launch behind it (a
// write and a read of 2 N bytes a row) took, and what they give: gate and up are rounded on their way into the unit, so what a prompt comes to does not hang on
// whether the tokens that happen to share its step are enough for tiles.  STORE, FLOAT: a product alone, with the bias in 32 bits, in bfloat16 or as it is.
// A product's results in bfloat16, each word of two or four columns a lane as it is, or of a gated unit
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int MI, int NI, int D, int EPI>
__global__ __launch_bounds__(256, 2) void tiles_kernel(const vmi_hy_linear_args p) {
  f32x4 bias[NI];
  vmi_tiles::tiles_product<vmi_tiles::Bf16, MI, NI, D>(
      p.x, p.ldx, p.w, p.M, p.N, p.K,
      [&](const vmi_tiles::Where& at) {
        if constexpr (EPI == VMI_HY_E_STORE) {
#pragma unroll
          for (int n = 0; n < NI; ++n)
            bias[n] = p.bias ? *reinterpret_cast<const f32x4*>(p.bias + min(at.s0 + at.wave * NI + n, at.SL - 1) * 16 + 4 * at.kc) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
      },
      [&](const f32x4(&acc)[NI][MI], const vmi_tiles::Where& at) {
        const int first = at.s0 * 16, wave_s = at.s0 + at.wave * NI, m = at.m0 + at.r16;
        auto stored = [&](int n, int i) {
          b16x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = EPI == VMI_HY_E_STORE ? (b16)(acc[n][i][r] + bias[n][r]) : (b16)acc[n][i][r];
          return __builtin_bit_cast(u32x2, o);
        };
        auto gated = [&](int n, int i) {
          typename Elem<b16>::v2 o;
#pragma unroll
          for (int r = 0; r < 2; ++r)
            o[r] = (b16)glu((float)(b16)acc[n][i][2 * r], (float)(b16)acc[n][i][2 * r + 1], p.scale, p.glu_alpha, p.glu_up);
          return __builtin_bit_cast(uint32_t, o);
        };
        if constexpr (EPI != VMI_HY_E_FLOAT) {
          if (EPI == VMI_HY_E_STORE || first + 64 * NI <= p.n_split) {   // (scalar)
            const bool wide = ((p.ldy & 7) | ((uintptr_t)p.y & 15)) == 0;
            vmi_tiles::lines_out<u32x2, MI, NI, false>(at, stored, [&](int row, int piece, const vmi_tiles::u32x4& v, int) {
              vmi_tiles::put_piece(at.m0 + row < p.M && first + 8 * piece < p.N, static_cast<b16*>(p.y) + (int64_t)(at.m0 + row) * p.ldy + first + 8 * piece, v, wide);
            });
            return;
          }
          if (first >= p.n_split) {
            const bool wide = ((p.ldy2 & 7) | ((uintptr_t)p.y2 & 15) | (p.n_split & 15)) == 0;
            vmi_tiles::lines_out<uint32_t, MI, NI, true>(at, gated, [&](int row, int piece, const vmi_tiles::u32x4& v, int) {
              vmi_tiles::put_piece(at.m0 + row < p.M && first + 16 * piece < p.N, static_cast<b16*>(p.y2) + (int64_t)(at.m0 + row) * p.ldy2 + ((first - p.n_split) >> 1) + 8 * piece, v, wide);
            });
            return;
          }
        }
#pragma unroll
        for (int n = 0; n < NI; ++n) {
          if (wave_s + n >= at.SL) break;   // (scalar)
          const int n0 = (wave_s + n) * 16, column = n0 + 4 * at.kc;
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            if (m + 16 * i >= p.M) continue;
            if constexpr (EPI == VMI_HY_E_FLOAT) {
              epilogue<b16, VMI_HY_E_FLOAT>(p, acc[n][i], m + 16 * i, column, n0, 0);
            } else if (n0 < p.n_split) {
              *reinterpret_cast<u32x2*>(static_cast<b16*>(p.y) + (int64_t)(m + 16 * i) * p.ldy + column) = stored(n, i);
            } else {
              *reinterpret_cast<uint32_t*>(static_cast<b16*>(p.y2) + (int64_t)(m + 16 * i) * p.ldy2 + ((column - p.n_split) >> 1)) = gated(n, i);
            }
          }
        }
      });
}

// Products of a group of matrices, a group a y of the grid, each with its own columns of x and of y (the per-head products of latent attention, of low ranks)
template <int MI, int NI, int D, int EPI>
__global__ __launch_bounds__(256, 2) void group_tiles_kernel(const vmi_hy_linear_args p) {
  const int grp = blockIdx.y;
  vmi_tiles::tiles_product<vmi_tiles::Bf16, MI, NI, D>(
      static_cast<const b16*>(p.x) + (int64_t)grp * p.x_gstride, p.ldx, static_cast<const b16*>(p.w) + (int64_t)grp * p.N * p.K, p.M, p.N, p.K,
      [](const vmi_tiles::Where&) {},
      [&](const f32x4(&acc)[NI][MI], const vmi_tiles::Where& at) {
        float g[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i)
          g[i] = EPI == VMI_HY_E_GATED ? sigmoid((float)static_cast<const b16*>(p.gate)[(int64_t)min(at.m0 + at.r16 + 16 * i, p.M - 1) * p.ldg + grp]) : 1.f;
        f32x4 bias[NI];
#pragma unroll
        for (int n = 0; n < NI; ++n)
          bias[n] = EPI == VMI_HY_E_STORE && p.bias ? *reinterpret_cast<const f32x4*>(p.bias + min(at.s0 + at.wave * NI + n, at.SL - 1) * 16 + 4 * at.kc) : f32x4{0.f, 0.f, 0.f, 0.f};
        b16* const y = static_cast<b16*>(p.y) + (int64_t)grp * p.y_gstride + at.s0 * 16;
        const bool wide = ((p.ldy & 7) | (p.y_gstride & 7) | ((uintptr_t)p.y & 15)) == 0;
        vmi_tiles::lines_out<u32x2, MI, NI, false>(
            at,
            [&](int n, int i) {
              b16x4 o;
#pragma unroll
              for (int r = 0; r < 4; ++r) o[r] = EPI == VMI_HY_E_GATED ? (b16)(acc[n][i][r] * g[i]) : (b16)(acc[n][i][r] + bias[n][r]);
              return __builtin_bit_cast(u32x2, o);
            },
            [&](int row, int piece, const vmi_tiles::u32x4& v, int) {
              vmi_tiles::put_piece(at.m0 + row < p.M && at.s0 * 16 + 8 * piece < p.N, y + (int64_t)(at.m0 + row) * p.ldy + 8 * piece, v, wide);
            });
      });
}

// Whether a group's products go to tiles: whole chunks of K, what the tiles' loads are aligned to, and more rows than plain_rows_kernel takes (all of ten groups below 65
// rows: 2.4 - 2.9 -> 2.9 - 3.8 us).  Not where K is four chunks at most and all tiles run at once, 64 rows or more each: nothing is beside a tile's ends then, and
// linear_kernel deals the rows finer.  Both over 246 products of 19 groups (2 to 64 matrices, K 64 to 512, N 64 to 4096, 65 to 4500 rows): this rule 0.1 per cent
// behind the better side in the mean, 4 at most; tiles always 1.2 and 14.  linear_kernel / tiles, us: 16 groups of K 128, N 512 97 / 300 / 900 / 2773 rows 4.0 / 5.3 / 12.1 / 28.7 -> 3.5 / 5.2 / 10.0
// / 24.4; of K 512, N 128 879 / 2773 8.8 / 27.6 -> 7.2 / 18.9; 8 of K 512, N 128 2260 11.1 -> 8.4; 2 of K 192, N 4096 900 13.2 -> 10.9.  Where the rule declines: 32 of K 128, N 512 177 rows 5.5 / 6.2; 4 of
// K 64, N 2048 354 5.4 / 6.2; 2 of K 192, N 4096 220 5.4 / 6.0.
static bool group_tiles_ahead(int M, int N, int K, int groups) {
  if (M <= 64) return false;
  const vmi_tiles::Tile& t = vmi_tiles::TILES[vmi_tiles::tiles_pick(M, N, K, groups)];
  return !(K <= 256 && t.mi >= 4 && (int64_t)vmi_tiles::tiles_grid(t, M, N) * groups <= 256);
}
bool group_tiles_fit(const vmi_hy_linear_args& p) {
  return p.groups > 1 && p.groups < 65536 && (p.N & 15) == 0 && (p.ldx & 7) == 0 && (p.x_gstride & 7) == 0 && p.x_gstride >= 0 && ((uintptr_t)p.x & 15) == 0 &&
         ((uintptr_t)p.w & 15) == 0 && vmi_tiles::tiles_fit(p.M, p.K, p.ldx) && group_tiles_ahead(p.M, p.N, p.K, p.groups);
}

template <int EPI, int I = 0>
static int launch_group_tiles_of(int pick, const vmi_hy_linear_args& p, hipStream_t st) {
  if constexpr (I < vmi_tiles::NTILES) {
    if (pick != I) return launch_group_tiles_of<EPI, I + 1>(pick, p, st);
    constexpr vmi_tiles::Tile T = vmi_tiles::TILES[I];
    hipLaunchKernelGGL((group_tiles_kernel<T.mi, T.ni, T.d, EPI>), dim3(vmi_tiles::tiles_grid(T, p.M, p.N), p.groups), dim3(256), 0, st, p);
    return launched("vmi_hy_linear");
  }
  return fail(VMI_HY_E_SHAPE, "vmi_hy_linear", "no such tile");
}

int launch_group_tiles(const vmi_hy_linear_args& p, hipStream_t st) {
  const int pick = vmi_tiles::tiles_pick(p.M, p.N, p.K, p.groups);
  return p.epilogue == VMI_HY_E_STORE ? launch_group_tiles_of<VMI_HY_E_STORE>(pick, p, st) : launch_group_tiles_of<VMI_HY_E_GATED>(pick, p, st);
}

// Whether tiles of our own end sooner than the library's product (hipBLASLt as PyTorch 2.10.0+rocm7.0 loads it: another version may move the line, never the result beyond the
// order of a sum).  Measured in bfloat16, weights that leave the last cache between two products from K 2048 on and others that stay.
//
// Alone, 5300 pairs of 48 to 9000 rows, K 256 to 12 288, N 256 to 16 384: ours / library's in the mean, from 5.6 million results on (below, nearly all of the library's time is its call:
// 19 us of host) and whole tiles of 256 columns: K 1024 to 2047 0.88 (8 of 207 more than 5 per cent behind), beyond 6144 1.07; other columns 0.74, 0.85 to K 4095, 0.96 to 6144 and 0.99 beyond.
// So not past K 6144 from 5.6 million results on, and whole columns up to 9 million, below K 2048 up to 15.  Whole columns between 5.6 and 9 million, K 2048 to 6144, 648 pairs by a grid and 596 by chance, ours / library's:
//   K up to 3072     always: 0.95 (20 of 376 more than 5 per cent behind, 1.17 at most, at sizes among others that are as far ahead)
//   beyond           0.99 (178 of 868, 1.23); so where the library's tiles, 256 x 128 as its times have them, leave a quarter of the compute units' turns empty, and the tiles' own costs promise 950 TFLOP/s (past K 4096
//                    1000), which is 0.92 (4 of 266, 1.10) and leaves 1.02 to the library.  N 2048, K 5120 2744 rows 0.85, 2929 0.92, 3173 to 3906 0.99 to 1.05, 4150 0.94, 4379 0.90; N 6144, K 5120 914 0.84, 1057 1.08, 1383 0.88.
// Not where few of the smallest tiles walk a long K each, which the library shares out (us, from here on the library's / ours: 64 rows, N 2048, K 6144 14.0 / 16.1; 140 24.4 / 22.4): measured again over 380 pairs of up to 128
// such tiles, now that results leave as lines, ours over the library's in the mean K 3072 0.93, 3584 and 4096 up to N 2048 0.96 (N 3072 1.17 and 1.02), 4608 and 5120 0.99 and 1.00 (1.11), 6144 1.15, 8192
// 1.31; and a call of the library's is 12 us more of host, which is what a short prompt waits for (62 rows, N 1024, K 3072 10.4 / 8.6 us, host 20 / 8).  Nor where tiles of 64 x 64 are just more than
// the chip has compute units for (300 rows, N 4096, K 8192 46 / 56; 600 rows, N 2048, K 6144 34 / 37), and past K 16 383.
static bool product_pays(int M, int N, int K) {
  const bool whole = N % 256 == 0;
  const int64_t results = (int64_t)M * N, least = (int64_t)((M + 31) / 32) * ((N + 63) / 64);
  if (results >= 5600000 && K > 6144) return false;
  if (whole && K >= 1024 && results >= (K >= 2048 ? 9000000 : 15000000)) return false;
  if (whole && results >= 5600000 && K > 3072) {
    auto turns = [&](int m, int n) { return ((int64_t)((M + m - 1) / m) * ((N + n - 1) / n) + 255) / 256; };   // of 256 compute units
    const int64_t least_turns = std::min(turns(256, 128), turns(128, 256));
    if (4 * results >= 3 * least_turns * 256 * 32768 ||
        2. * (double)results * K < (K <= 4096 ? .95e9 : 1e9) * vmi_tiles::tiles_cost(vmi_tiles::tiles_pick(M, N, K), M, N, K, 1))
      return false;
  }
  const bool shared = K > 4096 || (K > 3072 && N > 2048);   // (up to 4096 and 2048 nothing is to be had from sharing K out)
  if (K >= 3072 && ((shared && least <= 128) || (whole && N >= 2048 && results >= 1050000 && results < 2400000))) return false;
  return K < 16384;
}

// With the gated unit behind them (library and unit in a launch of its own / ours), 1930 pairs of 48 to 12 000 rows, K 512 to 16 384, N 1024 to 45 056: ours 0.86 of
// the time (K below 2048 0.74, 4096 0.85, 7168 0.90, beyond 0.95).  By K, results, and whether columns are whole tiles of 256, ours are ahead or level in
// every class but two past K 7168.  Where few of the smallest tiles walk a long K each 1.13 of 12 (76 rows, N 2048, K 16384 38 / 51), and where the library's largest
// tiles go round once, more than a third full, 1.03 of 86 (420 rows, N 20480, K 8192 142 / 174; 1200, 8192, 16384 275 / 328).
// What is left is single pairs that no size explains: below K 4096 8 of 927 are more than 5 per cent behind (1.11 at most), below 7168 45 of 450 (1.22; 6000 rows,
// N 40960, K 4096 1493 / 1712), beyond 76 of 455 (1.24), beside more of the like that are as far ahead (948, 40960, 4096 363 / 297).
// us: K 1024, N 6144 all gated 300 rows 13.0 / 8.5, 4500 66 / 58; K 2048, N 20480, 12288 of them gated, 140 rows 35 / 31, 2400 268 / 201.
static bool gated_whatever_rows(int K) { return K < 7168; }
static bool gated_pays(int M, int N, int K) {
  const int64_t results = (int64_t)M * N, least = (int64_t)((M + 31) / 32) * ((N + 63) / 64);
  return gated_whatever_rows(K) || (least > 128 && !(N % 256 == 0 && results >= 6000000 && results < 15000000));
}

template <int EPI, int I = 0>
static int launch_tiles(int pick, const vmi_hy_linear_args& p, hipStream_t st) {
  if constexpr (I < vmi_tiles::NTILES) {
    if (pick != I) return launch_tiles<EPI, I + 1>(pick, p, st);
    constexpr vmi_tiles::Tile T = vmi_tiles::TILES[I];
    hipLaunchKernelGGL((tiles_kernel<T.mi, T.ni, T.d, EPI>), dim3(vmi_tiles::tiles_grid(T, p.M, p.N)), dim3(256), 0, st, p);
    return launched("vmi_hy_linear_tiles");
  }
  return fail(VMI_HY_E_SHAPE, "vmi_hy_linear_tiles", "no such tile");
}

}  // namespace vmi_hybrid

using namespace vmi_hybrid;

extern "C" {

static bool linear_tiles_fit(int32_t N, int32_t K, int32_t n_split, int32_t dtype) {
  return dtype == VMI_HY_BF16 && N > 0 && K > 0 && n_split >= 0 && n_split < N && ((N | n_split) & 15) == 0 && (K & 63) == 0;
}

int32_t vmi_hy_linear_tiles_pay(int32_t M, int32_t N, int32_t K, int32_t n_split, int32_t dtype) {
  return M > 0 && linear_tiles_fit(N, K, n_split, dtype) && vmi_tiles::tiles_fit(M, K, K) && gated_pays(M, N, K);
}

int32_t vmi_hy_linear_tiles_only(int32_t N, int32_t K, int32_t n_split, int32_t dtype) { return linear_tiles_fit(N, K, n_split, dtype) && gated_whatever_rows(K); }

int32_t vmi_hy_tiles_pick(int32_t M, int32_t N, int32_t K, int32_t groups) {
  if (M <= 0 || N <= 0 || K <= 0 || groups <= 0 || (N & 15) || !vmi_tiles::tiles_fit(M, K, K)) return -1;
  return groups == 1 || group_tiles_ahead(M, N, K, groups) ? vmi_tiles::tiles_pick(M, N, K, groups) : -1;
}

int vmi_hy_linear_tiles(const vmi_hy_linear_args* a, void* stream) {
  static const char* who = "vmi_hy_linear_tiles";
  if (!a || !a->x || !a->w || !a->y || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->groups != 1 || a->dtype != VMI_HY_BF16 || a->x_kind != VMI_HY_X_ROWS ||
      (a->epilogue != VMI_HY_E_GLU && a->epilogue != VMI_HY_E_STORE_GLU) || (a->epilogue == VMI_HY_E_STORE_GLU && !a->y2))
    return fail(VMI_HY_E_ARG, who, "needs bfloat16 rows in one group and the gated unit behind all or some of the columns");
  vmi_hy_linear_args p = *a;
  if (p.epilogue == VMI_HY_E_GLU) p.y2 = p.y, p.ldy2 = p.ldy, p.n_split = 0;
  if ((p.N & 15) || (p.n_split & 15) || p.n_split < 0 || p.n_split > p.N || p.ldx < p.K || (p.ldx & 7) || !vmi_tiles::tiles_fit(p.M, p.K, p.ldx) ||
      (p.n_split && (p.ldy & 3)) || (p.ldy2 & 1) || ((uintptr_t)p.x & 15) || ((uintptr_t)p.w & 15) || (p.n_split && ((uintptr_t)p.y & 7)) || ((uintptr_t)p.y2 & 3))
    return fail(VMI_HY_E_SHAPE, who, "needs K % 64 == 0, N and n_split multiples of 16, 16-byte aligned rows of x, less than 4 GiB of them");
  DeviceScope dev(p.device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  return launch_tiles<VMI_HY_E_STORE_GLU>(vmi_tiles::tiles_pick(p.M, p.N, p.K), p, static_cast<hipStream_t>(stream));
}

int32_t vmi_hy_product_tiles_pay(int32_t M, int32_t N, int32_t K, int64_t ldx, int32_t dtype) {
  return dtype == VMI_HY_BF16 && M > 0 && N > 0 && K > 0 && (N & 15) == 0 && ldx >= K && (ldx & 7) == 0 && vmi_tiles::tiles_fit(M, K, ldx) && product_pays(M, N, K);
}

int vmi_hy_product_tiles(const vmi_hy_linear_args* a, void* stream) {
  static const char* who = "vmi_hy_product_tiles";
  if (!a || !a->x || !a->w || !a->y || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->groups != 1 || a->dtype != VMI_HY_BF16 || a->x_kind != VMI_HY_X_ROWS ||
      (a->epilogue != VMI_HY_E_STORE && a->epilogue != VMI_HY_E_FLOAT) || (a->bias && a->epilogue != VMI_HY_E_STORE))
    return fail(VMI_HY_E_ARG, who, "needs bfloat16 rows in one group, stored as they are (with a bias or none) or in 32 bits");
  const vmi_hy_linear_args& p = *a;
  if ((p.N & 15) || p.ldx < p.K || (p.ldx & 7) || !vmi_tiles::tiles_fit(p.M, p.K, p.ldx) || ((uintptr_t)p.x & 15) || ((uintptr_t)p.w & 15))
    return fail(VMI_HY_E_SHAPE, who, "needs K % 64 == 0, N a multiple of 16, 16-byte aligned rows of x, less than 4 GiB of them");
  if (p.epilogue == VMI_HY_E_STORE ? (p.ldy < p.N || (p.ldy & 3) || ((uintptr_t)p.y & 7) || ((uintptr_t)p.bias & 15))
                                   : (p.n_out <= 0 || p.n_out > p.N || p.ldy < p.n_out || ((uintptr_t)p.y & 15)))
    return fail(VMI_HY_E_SHAPE, who, "needs room for a row's columns in y, y and bias aligned to four elements of theirs");
  DeviceScope dev(p.device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  const int pick = vmi_tiles::tiles_pick(p.M, p.N, p.K);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  return p.epilogue == VMI_HY_E_STORE ? launch_tiles<VMI_HY_E_STORE>(pick, p, st) : launch_tiles<VMI_HY_E_FLOAT>(pick, p, st);
}

}  // extern "C"
