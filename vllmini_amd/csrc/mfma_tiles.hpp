// Products of many rows, y = x W^T, in 16-bit elements: x as rows, W as the tiles the linear layers pack ([N / 16][K / 32][64 lanes][8]).
//
// A workgroup's tile is 16 MI rows x 64 NI columns; four waves own 16 NI columns each and ALL of its rows.  So a wave's weights are nobody else's: they go from
// memory straight to registers as they lie, one contiguous KiB a k-step, 64 columns of K ahead.  x goes through LDS: whole 128-byte lines in, through registers, two
// buffers and one barrier per 64 columns of K; 16-byte piece c of row r lies at c ^ (r & 7) of its line, so that eight consecutive lanes, eight rows of one piece, meet in no
// bank.  KS = 2: two groups of four waves take half of K each (few tiles, long K), their results meet in LDS.
//
// Bound by the matrix cores' and the waves' issue together, 4.1 to 5 TFLOP/s a compute unit (the card 1.24 PFLOP/s at 8192^3, the vendor's kernels 1.34; both operands in LDS, 2 x 2
// waves: 0.82), and by how the tiles share the chip out (tiles_pick).  2770 rows, N 12288, K 2048 131 us (vendor 132 - 138), N 2048, K 6144 69 (68 - 76), N 2048, K 2048 29
// (27); 4500 rows, N 10240, K 1024 106 (81 - 109); 3200 rows, N 20480, K 2048 240 (270 - 290); 6300 rows, N 3072, K 768 43 (40 - 49): level, and what follows
// a product (bias, GELU, gated unit, residual) rides along.  Two row groups of four waves over one tile (256 x 256, weights from L1 a second time): 0.83 of it.  32x32x16
// matrix instructions: 0.95.  Tiles of 192 and 256 rows in one wave's registers spill.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vmi_tiles {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Half {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(const v8& a, const v8& b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
struct Bf16 {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(const v8& a, const v8& b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

template <int MI, int NI, int KS>
constexpr size_t tiles_lds() {
  const size_t x = (size_t)KS * 2 * 16 * MI * 128, parts = KS == 2 ? (size_t)16 * MI * 64 * NI * 4 : 0;
  return x > parts ? x : parts;
}

// The product of this workgroup's tile; early(m, s, SL) asks for what finish will read, behind the first requests of the product; finish(acc, m, s, SL) gets a lane's results, acc[n][i] = columns 16 (s + n) + 4 (lane / 16) .. + 3 of row m + 16 i, and does not look at
// slabs from SL or rows from M on.  K % 64 == 0, N % 16 == 0, x and ldx 16-byte aligned, a matrix of x below 4 GiB.
template <class H, int MI, int NI, int KS, bool PRIO, class Early, class Finish>
__device__ __forceinline__ void tiles_product(const void* x, int64_t ldx, const void* w, int M, int N, int K, unsigned char* smem, Early&& early, Finish&& finish) {
  using V8 = typename H::v8;
  constexpr int BM = 16 * MI, BN = 64 * NI, ST = BM * 128, XU = BM * 8 / 256;   // 16-byte pieces of x a thread brings
  const int tid = threadIdx.x & 255, lane = tid & 63, kc = lane >> 4, r16 = lane & 15;
  const int g = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* xs = smem + g * 2 * ST;
  const int SL = N >> 4, NB = (N + BN - 1) / BN, MB = (M + BM - 1) / BM;
  // workgroups go to the eight dies in turn: each die takes a run of whole columns of tiles, whose weights it then reads once
  const int all = NB * MB, die = (int)blockIdx.x & 7, tile = die * (all >> 3) + min(die, all & 7) + ((int)blockIdx.x >> 3);
  const int m0 = tile % MB * BM, s0 = tile / MB * 4 * NI + wave * NI;
  const int nkb = K >> 6, per = (nkb + KS - 1) / KS, k0 = g * per, k1 = min(nkb, k0 + per);
  // (rows past the last, slabs past the last and steps past the end are those again: no lane-wise condition around a load)
  const char* xb = static_cast<const char*>(x);
  uint32_t xo[XU];
#pragma unroll
  for (int i = 0; i < XU; ++i) xo[i] = (uint32_t)min(m0 + (tid >> 3) + 32 * i, M - 1) * (uint32_t)(ldx * 2) + (uint32_t)((tid & 7) ^ ((tid >> 3) & 7)) * 16;
  const char* wb[NI];
#pragma unroll
  for (int n = 0; n < NI; ++n) wb[n] = static_cast<const char*>(w) + (int64_t)min(s0 + n, SL - 1) * (K >> 5) * 1024;
  V8 xr[XU], wr[2][2][NI];
  auto load_x = [&](int kb) {
    const uint32_t at = (uint32_t)min(kb, nkb - 1) * 128;
#pragma unroll
    for (int i = 0; i < XU; ++i) xr[i] = *reinterpret_cast<const V8*>(xb + (xo[i] + at));
  };
  auto load_w = [&](V8(&to)[2][NI], int kb) {
    const int k = min(kb, nkb - 1);
#pragma unroll
    for (int n = 0; n < NI; ++n)
#pragma unroll
      for (int j = 0; j < 2; ++j) to[j][n] = *reinterpret_cast<const V8*>(wb[n] + k * 2048 + (uint32_t)(j * 1024 + lane * 16));
  };
  auto put_x = [&](int s) {
#pragma unroll
    for (int i = 0; i < XU; ++i) *reinterpret_cast<V8*>(xs + s * ST + i * 4096 + tid * 16) = xr[i];
  };
  const int frag = r16 * 128 + ((kc ^ (r16 & 7)) * 16);
  f32x4 acc[NI][MI];
#pragma unroll
  for (int n = 0; n < NI; ++n)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[n][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  load_x(k0);
  load_w(wr[0], k0);
  put_x(0);
  load_x(k0 + 1);
  if (KS == 1 || g == 0) early(m0 + r16, s0, SL);
  __syncthreads();
  auto chunk = [&](int kb, int s, V8(&cur)[2][NI], V8(&nxt)[2][NI]) {
    load_w(nxt, kb + 1);
    put_x(s ^ 1);   // (every wave has passed the barrier behind its reads of that buffer)
    load_x(kb + 2);
    V8 f[2][MI];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i) f[j][i] = *reinterpret_cast<const V8*>(xs + s * ST + (frag ^ (j * 64)) + i * 2048);
    if (KS == 1 || kb < k1) {   // (scalar: an odd number of chunks)
      if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int n = 0; n < NI; ++n) acc[n][i] = H::mma(cur[j][n], f[j][i], acc[n][i]);
      if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
    }
    // requests, then x on, then the fragments three ahead of the products that take them
    __builtin_amdgcn_sched_group_barrier(0x020, 2 * NI, 0);
    __builtin_amdgcn_sched_group_barrier(0x200, XU, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, XU, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
    for (int i = 0; i < 2 * MI - 3; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, NI, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 3 * NI, 0);
    __syncthreads();
  };
  for (int i = 0; i < per; i += 2) {
    chunk(k0 + i, 0, wr[0], wr[1]);
    if (i + 1 < per) chunk(k0 + i + 1, 1, wr[1], wr[0]);
  }
  if constexpr (KS == 2) {
    f32x4* part = reinterpret_cast<f32x4*>(smem) + wave * NI * MI * 64 + lane;
    if (g == 1) {
#pragma unroll
      for (int n = 0; n < NI; ++n)
#pragma unroll
        for (int i = 0; i < MI; ++i) part[(n * MI + i) * 64] = acc[n][i];
    }
    __syncthreads();
    if (g == 1) return;
#pragma unroll
    for (int n = 0; n < NI; ++n)
#pragma unroll
      for (int i = 0; i < MI; ++i) acc[n][i] += part[(n * MI + i) * 64];
  }
  finish(acc, m0 + r16, s0, SL);
}

// ---- which tile -----------------------------------------------------------------------------------------------------------------
struct Tile {
  int mi, ni, ks;
  bool prio;            // the products at a raised wave priority: ahead where waves of two workgroups share a compute unit's matrix cores
  float alone, beside;  // us per 64 columns of K: one workgroup a compute unit, and a workgroup's share of a full one
};
// fitted to 258 products of 100 to 8192 rows, N 512 to 24576, K 768 to 12288
constexpr Tile TILES[] = {{8, 4, 1, false, .90f, .83f}, {8, 3, 1, false, .77f, .76f}, {6, 4, 1, true, .85f, .61f}, {6, 3, 1, false, .64f, .51f}, {6, 2, 1, false, .47f, .42f},
                          {8, 2, 1, false, .50f, .50f}, {4, 2, 1, false, .44f, .30f}, {4, 2, 2, false, .39f, .34f}, {4, 1, 2, false, .27f, .22f}};
constexpr int NTILES = sizeof(TILES) / sizeof(TILES[0]);

// us, as the chip's tiles are dealt
inline float tiles_cost(int i, int M, int N, int K) {
  const Tile& t = TILES[i];
  const int64_t n = (int64_t)((M + 16 * t.mi - 1) / (16 * t.mi)) * ((N + 64 * t.ni - 1) / (64 * t.ni)), share = (n + 255) / 256;
  return (share == 1 ? t.alone : share * t.beside) * ((float)(K >> 6) + (t.ks == 2 ? 9.5f : 6.f));
}

// The tile whose largest share of a compute unit ends first: so many tiles one behind the other, each 64 columns of K at a time and as long as 6 such at its ends (9.5
// where two halves meet).  On average 0.5 per cent behind the best of the list over those 258 products, 11 at most.  (us, 128 x 256 / 128 x 192 / 96 x 256 / 64 x 128: 2770
// rows, N 2048, K 6144 86 / 69 / 75 / 89, of 176 / 242 / 232 / 704 tiles; 2100 rows, N 768, K 768 16 / 13 / 13 / 7.)
inline int tiles_pick(int M, int N, int K) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < NTILES; ++i) {
    const float cost = tiles_cost(i, M, N, K);
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}
inline unsigned tiles_grid(const Tile& t, int M, int N) { return (unsigned)((M + 16 * t.mi - 1) / (16 * t.mi)) * (unsigned)((N + 64 * t.ni - 1) / (64 * t.ni)); }
inline bool tiles_fit(int M, int K, int64_t ldx) { return (K & 63) == 0 && (int64_t)M * ldx * 2 < (int64_t)1 << 32; }

}  // namespace vmi_tiles
