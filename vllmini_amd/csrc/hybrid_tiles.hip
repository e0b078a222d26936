// Products of many rows in bfloat16 with the gated unit behind them (mfma_tiles.hpp), include/vmi_hybrid.h: vmi_hy_linear_tiles.
#include "hybrid_common.hpp"
#include "hybrid_linear.hpp"
#include "mfma_tiles.hpp"

namespace vmi_hybrid {

// Columns below n_split as they are, the others, interleaved (gate, up), through the gated unit: what a product and an elementwise launch behind it (a
// write and a read of 2 N bytes a row) took, and what they give: gate and up are rounded on their way into the unit, so what a prompt comes to does not hang on
// which side tiles_pay finds ahead for the tokens that happen to share its step.
template <int MI, int NI, int D>
__global__ __launch_bounds__(256, 2) void tiles_kernel(const vmi_hy_linear_args p) {
  const int kc = (threadIdx.x & 63) >> 4;
  vmi_tiles::tiles_product<vmi_tiles::Bf16, MI, NI, D>(
      p.x, p.ldx, p.w, p.M, p.N, p.K, [](int, int, int) {},
      [&](const f32x4(&acc)[NI][MI], int m, int s, int SL) {
#pragma unroll
        for (int n = 0; n < NI; ++n) {
          if (s + n >= SL) break;   // (scalar)
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            f32x4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = (float)(b16)acc[n][i][r];
            if (m + 16 * i < p.M) epilogue<b16, VMI_HY_E_STORE_GLU>(p, v, m + 16 * i, (s + n) * 16 + 4 * kc, (s + n) * 16, 0);
          }
        }
      });
}

// Whether tiles of our own with the unit behind them end sooner than the library's product and the unit in a launch of its own.  Ours are ahead where the
// library's tiles of 256 x 256 leave part of the chip idle or rows are few, behind where they fill it (they take 0.74 of ours' time then).  Both sides as their tiles share
// the chip out; the library's (hipBLASLt as PyTorch 2.10.0+rocm7.0 loads it: another version may move the line, never the result) fitted to 80 products of 48 to 8192 rows, K 1024 to 4096, N 6144 to 24576, 9 per cent off in the mean, and the rule's picks within 0.6 per
// cent of the better side in the mean, 11 at most.  Library + unit / ours in us, cold weights: K 1024, N 6144 all gated 300 rows 14.9 / 10.4, 1500 36.6 / 24.3, 4500
// 65.8 / 65.3; K 2048, N 20480, 12288 of them gated, 100 rows 34.4 / 27.0, 1500 113 / 129, 3200 301 / 257, 8192 530 / 639; K 4096, N 24576 48 49.4 / 44.6, 2400 387 / 440.
static bool tiles_pay(int M, int N, int K, int n_split) {
  struct Library {
    int bm, bn;
    float chunk, ends;
  };
  constexpr Library LIBRARY[] = {{256, 256, 1.38f, 4.1f}, {128, 256, .86f, 4.6f}, {128, 128, .82f, 2.f}, {64, 128, .66f, 2.1f}, {64, 64, .34f, 5.6f}};
  float least = 0.f;
  for (const Library& t : LIBRARY) {
    const int64_t n = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const float cost = (float)((n + 255) / 256) * t.chunk * (float)(K >> 6) + t.ends;
    if (&t == LIBRARY || cost < least) least = cost;
  }
  return vmi_tiles::tiles_cost(vmi_tiles::tiles_pick(M, N, K), M, N, K) < least + .76f + (float)M * (float)(N - n_split) / 1.26e6f;
}

template <int I = 0>
static int launch_tiles(int pick, const vmi_hy_linear_args& p, hipStream_t st) {
  if constexpr (I < vmi_tiles::NTILES) {
    if (pick != I) return launch_tiles<I + 1>(pick, p, st);
    constexpr vmi_tiles::Tile T = vmi_tiles::TILES[I];
    hipLaunchKernelGGL((tiles_kernel<T.mi, T.ni, T.d>), dim3(vmi_tiles::tiles_grid(T, p.M, p.N)), dim3(256), 0, st, p);
    return launched("vmi_hy_linear_tiles");
  }
  return fail(VMI_HY_E_SHAPE, "vmi_hy_linear_tiles", "no such tile");
}

}  // namespace vmi_hybrid

using namespace vmi_hybrid;

extern "C" {

int32_t vmi_hy_linear_tiles_pay(int32_t M, int32_t N, int32_t K, int32_t n_split, int32_t dtype) {
  return dtype == VMI_HY_BF16 && M > 0 && N > 0 && K > 0 && n_split >= 0 && n_split < N && ((N | n_split) & 15) == 0 && vmi_tiles::tiles_fit(M, K, K) &&
         tiles_pay(M, N, K, n_split);
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
  return launch_tiles(vmi_tiles::tiles_pick(p.M, p.N, p.K), p, static_cast<hipStream_t>(stream));
}

}  // extern "C"
