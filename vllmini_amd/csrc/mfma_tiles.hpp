// Products of many rows, y = x W^T, in 16-bit elements: x as rows, W as the tiles the linear layers pack ([N / 16][K / 32][64 lanes][8]).
//
// A workgroup's tile is 16 MI rows x 64 NI columns; four waves own 16 NI columns each and ALL of its rows.  So a wave's weights are nobody else's: they go from
// memory straight to registers as they lie, one contiguous KiB a k-step.  x goes from memory straight into LDS (buffer loads that end there), whole 128-byte lines, a place of 64
// columns of K a chunk; 16-byte piece c of row r lies at c ^ (r & 7) of its line, so that the lanes of one read meet in no bank.  D places are in flight, D - 1 chunks ahead, with
// one barrier a chunk, and requests, reads of x and products are dealt over the chunk's steps one by one.
//
// What bounds it: tiles that have a compute unit to themselves the latency of memory, so those stay four chunks deep (300 rows, N 2048, K 6144 23.8 -> 19.3 us, the vendor's
// kernels 28.5; 700 rows, N 768, K 3072 14.6 -> 11.8; 120 rows, N 2304, K 768 6.5 -> 4.9); a full chip L2 and the matrix cores at the clock that their power leaves (2773 rows, N 12288,
// K 2048: 2.0 GHz, 47 per cent of their cycles): the order of tiles took 0.67 GB of misses in L2 to 0.41 there (143 -> 139 us, vendor 135 - 143; N 2048, K 6144 69 -> 63, 73) and 6146
// rows, N 3072, K 768 with GELU from 52 to 40.  x through registers, two buffers: 18 per cent behind on average over 454 products, a quarter below 300 rows.  Taken back: eight
// waves over 256 x 256 or 192 x 256 with both operands in LDS (level with these at 2773 rows, 0.97 of them at 8192^3), the same in four waves of 128 x 128 (level); a
// workgroup for several tiles, which asks for the next one's first chunks behind the present one's last (within 2 per cent); K over two groups of waves (behind four chunks ahead).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

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

// Where a tile's results are: rows m0 on, slabs of 16 columns s0 on; a lane holds acc[n][i] = columns 16 (s0 + wave NI + n) + 4 kc .. + 3 of row m0 + 16 i + r16.  Slabs from SL and
// rows from M on are none.  lds: two places of 2 KiB MI, free once every wave is past a barrier.
struct Where {
  int m0, s0, SL, wave, kc, r16;
  unsigned char* lds[2];
};

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Results of 16 bits on their way out, as whole lines: 32 rows of the tile at a time through LDS.  pack(n, i): what a lane has of slab n, tile i, eight bytes (four columns) or
// four (two, behind a gated unit), all of it FIRST where that is work (between two barriers there is nothing but LDS then); put(row, piece, v, k): sixteen bytes from 16 piece on
// of a row of the tile, the k-th of this lane, neighbours of a row in neighbouring lanes: NI pieces of every 32 rows, one of (threadIdx.x + 256 j) / PIECES, % PIECES.
// What bounds it is L2, which takes as long for 32 bytes of a line as for 64 or 128: as the lanes hold them, a store would leave 32 bytes of each of 16 lines (16 behind a gated unit), and
// products over a short K spent a third of their time on it.  us before / now: 6400 rows, K 768 in halves N 2304 29.3 / 24.7, N 768 with a residual 17.0 / 13.7, K 3072 37.9 / 32.4; gated, bfloat16
// 2773 rows, N 12288, K 2048 128 / 116, 4600, 6144, 1024 58 / 51; without any stores 6400 rows, N 2304 take 18.4.
template <class Word, int MI, int NI, bool FIRST, class Pack, class Put>
__device__ __forceinline__ void lines_out(const Where& at, Pack&& pack, Put&& put) {
  constexpr int PIECES = NI * (int)sizeof(Word), BYTES = 16 * PIECES, ALL = 32 * PIECES;
  // (a row's pieces in another order for each of eight rows, or rows an odd number of pieces apart: lanes of one access meet in no bank)
  constexpr bool TURN = sizeof(Word) == 8;
  constexpr int ROW = TURN ? BYTES : BYTES + 16;
  static_assert(32 * ROW <= MI * 2048 && MI % 2 == 0);
  auto landed = []() {   // (a fence would wait for the stores as well)
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  Word words[FIRST ? MI : 1][NI];
  if constexpr (FIRST) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int n = 0; n < NI; ++n) words[i][n] = pack(n, i);
  }
  landed();
#pragma unroll
  for (int t = 0; t < MI / 2; ++t) {
    unsigned char* const b = at.lds[t & 1];
#pragma unroll
    for (int n = 0; n < NI; ++n)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 16 * h + at.r16, byte = (at.wave * NI + n) * 4 * (int)sizeof(Word) + at.kc * (int)sizeof(Word), piece = byte >> 4;
        *reinterpret_cast<Word*>(b + row * ROW + (TURN ? piece ^ (row & 7) : piece) * 16 + (byte & 15)) = FIRST ? words[FIRST ? 2 * t + h : 0][n] : pack(n, 2 * t + h);
      }
    landed();
#pragma unroll
    for (int j = 0; j < (ALL + 255) / 256; ++j) {
      const int u = (int)threadIdx.x + 256 * j, row = u / PIECES, piece = u - row * PIECES;
      if (ALL % 256 == 0 || u < ALL) put(32 * t + row, piece, *reinterpret_cast<const u32x4*>(b + row * ROW + (TURN ? piece ^ (row & 7) : piece) * 16), t * ((ALL + 255) / 256) + j);
    }
  }
}
// The same without LDS and barriers, in sixteen bytes of half a line: two slabs' neighbouring columns meet in a lane, whose (lane / 16) even ones keep slab n, odd ones n + 1.  NI even.
template <int MI, int NI, class Pack, class Put>
__device__ __forceinline__ void pairs_out(const Where& at, Pack&& pack, Put&& put) {
  static_assert(NI % 2 == 0);
#pragma unroll
  for (int n = 0; n < NI; n += 2)
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const u32x2 a = pack(n, i), b = pack(n + 1, i);
      const auto l = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), h = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
      put(16 * i + at.r16, (at.wave * NI + n + (at.kc & 1)) * 2 + (at.kc >> 1), u32x4{l[0], h[0], l[1], h[1]}, 0);
    }
}
// sixteen bytes of results, where this lane's are any; wide: rows of y and where they begin are aligned to as many, else to four (the scalar condition outside: inside the other one it is a branch more)
__device__ __forceinline__ void put_piece(bool on, void* y, const u32x4& v, bool wide) {
  if (wide) {   // (scalar)
    if (on) *static_cast<u32x4*>(y) = v;
  } else {
    if (on) {
#pragma unroll
      for (int r = 0; r < 4; ++r) static_cast<uint32_t*>(y)[r] = v[r];
    }
  }
}

// The product of this workgroup's tile; early(at) asks for what finish(acc, at) will read, behind the first requests of the product.
// K % 64 == 0, N % 16 == 0, x and ldx 16-byte aligned, a matrix of x below 4 GiB.
template <class H, int MI, int NI, int D, class Early, class Finish>
__device__ __forceinline__ void tiles_product(const void* x, int64_t ldx, const void* w, int M, int N, int K, Early&& early, Finish&& finish) {
  using V8 = typename H::v8;
  static_assert(D >= 2 && D <= 4, "a place a chunk, by name");
  constexpr int BM = 16 * MI, BN = 64 * NI, ST = BM * 128, XU = BM * 8 / 256;   // 16-byte pieces of x a thread brings
  constexpr int AHEAD = 4, STEPS = 2 * MI, ASKS = XU + 2 * NI, PER = (ASKS + STEPS - 1) / STEPS;
  static_assert(STEPS >= AHEAD, "fragments of one chunk");
  static_assert(PER == 1, "a barrier of the scheduler between any two requests of the walk");
  // (arrays by name: only so does the compiler know that a read of one does not wait for what is on its way into another)
  __shared__ __attribute__((aligned(1024))) unsigned char xs0[ST], xs1[ST], xs2[D > 2 ? ST : 1], xs3[D > 3 ? ST : 1];
  unsigned char* const xs[4] = {xs0, xs1, xs2, xs3};
  const int tid = threadIdx.x, lane = tid & 63, kc = lane >> 4, r16 = lane & 15, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int SL = N >> 4, NB = (N + BN - 1) / BN, MB = (M + BM - 1) / BM, nkb = K >> 6;
  // workgroups go to the eight dies in turn: each die takes a run of tiles, 1024 rows of x down and then the next columns, so that the tiles of a die that are under way
  // together share their rows and weights in its L2
  constexpr int DOWN = 1024 / BM;
  const int all = NB * MB, die = (int)blockIdx.x & 7, tile = die * (all >> 3) + min(die, all & 7) + ((int)blockIdx.x >> 3);
  // (a division leaves a scalar's value in a vector register: said here, or the compiler may keep what follows from it there, and ask for weights lane by lane)
  const int band = __builtin_amdgcn_readfirstlane(tile / (DOWN * NB)), in = tile - band * DOWN * NB, rows = min(DOWN, MB - band * DOWN), col = __builtin_amdgcn_readfirstlane(in / rows);
  const int m0 = (band * DOWN + in - col * rows) * BM, s0 = col * 4 * NI + wave * NI;
  // (rows past the last, slabs past the last and chunks past the end are those again: no lane-wise condition around a load)
  const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(x), 0, -1, 0x20000);
  uint32_t xo[XU], wo[NI];
#pragma unroll
  for (int i = 0; i < XU; ++i) xo[i] = (uint32_t)min(m0 + (tid >> 3) + 32 * i, M - 1) * (uint32_t)(ldx * 2) + (uint32_t)((tid & 7) ^ ((tid >> 3) & 7)) * 16;
  const int first = min(s0, SL - 1);
  const __amdgpu_buffer_rsrc_t wb =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(w)) + (int64_t)first * (K >> 5) * 1024, 0, -1, 0x20000);
#pragma unroll
  for (int n = 0; n < NI; ++n) wo[n] = (uint32_t)(min(s0 + n, SL - 1) - first) * (uint32_t)(K >> 5) * 1024;
  V8 wr[D][2][NI], f[AHEAD];
  // request i of chunk kb, which goes to place d: x first, which every wave waits for
  auto ask = [&](int i, int d, int kb) {
    if (i < XU) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xb, (__attribute__((address_space(3))) void*)(xs[d] + i * 4096 + wave * 1024), 16, xo[i], kb * 128, 0, 0);
    } else if (i < ASKS) {
      const int n = (i - XU) >> 1, j = (i - XU) & 1;
      wr[d][j][n] = __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(wb, lane * 16 + j * 1024, wo[n] + (uint32_t)kb * 2048, 0));
    }
  };
  const int frag = r16 * 128 + ((kc ^ (r16 & 7)) * 16);
  auto read = [&](const unsigned char* from, int q) { return *reinterpret_cast<const V8*>(from + (frag ^ (q / MI * 64)) + q % MI * 2048); };
  f32x4 acc[NI][MI];
#pragma unroll
  for (int n = 0; n < NI; ++n)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[n][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The x of the next chunk is there for every wave: this one has waited for all it asked for before that chunk's weights, the BEHIND whole chunks after those left out
  // (s_waitcnt counts in order; the barrier is the plain one, a fence would wait for all of x that is on its way)
  auto x_landed = [](auto behind) {
    constexpr int V = decltype(behind)::value * ASKS + 2 * NI;
    static_assert(V < 64, "vmcnt has six bits");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70 | (V & 15) | (V >> 4 << 14));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // (the counts above are of requests in this order, and to the scheduler requests into LDS and into registers have nothing to do with each other)
#pragma unroll
  for (int d = 0; d < D - 1; ++d) {
#pragma unroll
    for (int i = 0; i < ASKS; ++i) {
      ask(i, d, min(d, nkb - 1));
      if (i == XU - 1 || i == ASKS - 1) __builtin_amdgcn_sched_barrier(0);
    }
  }
  const Where at{m0, col * 4 * NI, SL, wave, kc, r16, {xs0, xs1}};
  early(at);
  x_landed(std::integral_constant<int, D - 2>{});
  // The chunk in place d, and chunk kb on its way into the place of the one before (whose readers have all passed the barrier): steps of one fragment of x, which was asked
  // for AHEAD steps before, against the wave's NI of W, and its share of the requests.  A chunk that is none is zeros, x and W
  auto chunk = [&](auto more, int d, int kb, bool on) {
    auto fragment = [&](int q) { return read(xs[d], q); };
    if (!on) {   // (scalar)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int n = 0; n < NI; ++n) wr[d][j][n] = V8{};
    }
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) f[q] = fragment(q);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < STEPS; ++q) {
      if constexpr (decltype(more)::value) {
#pragma unroll
        for (int i = 0; i < PER; ++i) ask(q * PER + i, (d + D - 1) % D, kb);
      }
      __builtin_amdgcn_sched_barrier(0);
      const V8 now = on ? f[q % AHEAD] : V8{};   // (here and not where it is read, or every read is waited for at once)
#pragma unroll
      for (int n = 0; n < NI; ++n) acc[n][q % MI] = H::mma(wr[d][q / MI][n], now, acc[n][q % MI]);
      if (q + AHEAD < STEPS) f[q % AHEAD] = fragment(q + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr std::true_type asking{};
  constexpr std::false_type asked{};
  int c = 0;
  for (; c + D < nkb; c += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      chunk(asking, d, min(c + d + D - 1, nkb - 1), true);
      x_landed(std::integral_constant<int, D - 2>{});
    }
  }
  // the last D places, 1 to D of them chunks (without a branch around a product, whose accumulators would change registers)
  chunk(asking, 0, nkb - 1, true);
  auto rest = [&](auto dd) {
    constexpr int d = decltype(dd)::value;
    if constexpr (d < D) {
      x_landed(std::integral_constant<int, (d < D ? D - 1 - d : 0)>{});
      chunk(asked, d, 0, c + d < nkb);
    }
  };
  rest(std::integral_constant<int, 1>{}), rest(std::integral_constant<int, 2>{}), rest(std::integral_constant<int, 3>{});
  finish(acc, at);
}

// ---- which tile -----------------------------------------------------------------------------------------------------------------
struct Tile {
  int mi, ni, d;
  float alone, beside;  // us per 64 columns of K: one workgroup a compute unit, and a workgroup's share of a full one
  float ends;           // ... as many of which its ends take
};
// fitted to 1080 products of 33 to 8192 rows, N 256 to 45 056, K 256 to 16 384, weights in the last cache and not
constexpr Tile TILES[] = {{8, 4, 2, .836f, .727f, 6.9f}, {8, 3, 2, .884f, .594f, 5.5f}, {8, 3, 4, .630f, .715f, 7.7f}, {6, 3, 2, .680f, .483f, 4.4f},
                          {6, 2, 2, .545f, .375f, 3.0f}, {6, 2, 4, .431f, .581f, 5.0f}, {8, 2, 2, .590f, .445f, 3.8f}, {8, 2, 4, .448f, 1.009f, 9.9f},
                          {4, 2, 2, .452f, .312f, 2.4f}, {4, 2, 4, .336f, .354f, 4.6f}, {4, 1, 4, .177f, .192f, 6.3f}, {2, 1, 2, .240f, .165f, 1.3f},
                          {2, 1, 4, .148f, .129f, 5.1f}};
constexpr int NTILES = sizeof(TILES) / sizeof(TILES[0]);

// us, as the chip's tiles are dealt
inline float tiles_cost(int i, int M, int N, int K, int groups) {
  const Tile& t = TILES[i];
  const int64_t n = (int64_t)((M + 16 * t.mi - 1) / (16 * t.mi)) * ((N + 64 * t.ni - 1) / (64 * t.ni)) * groups, share = (n + 255) / 256;
  const int chunks = ((K >> 6) + t.d - 1) / t.d * t.d;
  return 2.f + (share == 1 ? t.alone : share * t.beside) * ((float)chunks + t.ends);
}

// The tile whose largest share of a compute unit ends first: so many tiles one behind the other, each 64 columns of K at a time and as long as `ends` such at its ends.  On
// average 0.7 per cent behind the best of the list over those products.  (us, 128 x 256 / 128 x 192, four chunks / 96 x 128, four / 32 x 64, four: 2773 rows, N 2048,
// K 6144 81 / 63 / 75 / 190; 300 rows, the same 70 / 46 / 34 / 23 and 64 x 64 19.)
inline int tiles_pick(int M, int N, int K, int groups = 1) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < NTILES; ++i) {
    const float cost = tiles_cost(i, M, N, K, groups);
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}
inline unsigned tiles_grid(const Tile& t, int M, int N) { return (unsigned)((M + 16 * t.mi - 1) / (16 * t.mi)) * (unsigned)((N + 64 * t.ni - 1) / (64 * t.ni)); }
inline bool tiles_fit(int M, int K, int64_t ldx) { return (K & 63) == 0 && (int64_t)M * ldx * 2 < (int64_t)1 << 32; }

}  // namespace vmi_tiles
